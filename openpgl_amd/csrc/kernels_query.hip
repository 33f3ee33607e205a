// Batched guiding queries on gfx950: for each query, region lookup (kd walk
// plus the stochastic KNN pick), parallax shift of the region mixture to the
// query position, product with the cosine lobe (surface) or the 3-lobe
// Henyey-Greenstein representation (volume), one sample and its pdf.
//
// A quad of four lanes per query, each lane holding the products of a quarter
// of the components in registers between the integral, the CDF walk and the
// pdf (surface); the region data (4 KiB per region) stays L2/MALL resident
// while queries stream.
//
// Reference behaviour: Field::getRegion field/Field.h:109-145,
// SurfaceVolumeField::init*SamplingDistribution field/SurfaceVolumeField.h:50-85,
// VMMSurfaceSamplingDistribution.h:37-97, VMMVolumeSamplingDistribution.h:37-123.
#include <hip/hip_runtime.h>

#include "common.h"
#include "kernels.h"
#include "query_math.h"

namespace pglgpu {

// The four lanes of a quad (lanes 4i .. 4i + 3 of a wave) work on one query:
// lane q owns the components k = 4j + q (j < 8), so a query's component
// loops take a quarter of the serial steps and the component parameters of
// a region are read by four lanes at once.  Every lane of a quad runs the
// same control flow (the query decides it), so the quad sums below see four
// active lanes.
//
// Bound by the vector unit: the shift, product and pdf of a component are
// about 150 instructions, most of them correctly rounded divisions and square
// roots.  The component loops run over the groups that any query of the wave
// uses, two groups per branch (a branch per component serialised their chains);
// divisions by the same number share its reciprocal, and divisions and roots
// whose operands are far from the ends of the exponent range go without the
// scaling steps.  A component is read as two 16-byte loads of its region's
// query form (seven loads of one word each, from as many cache lines, took as
// long as the arithmetic).  2.07 M surface queries on 400 regions: 463 us at
// first, 378 with the arithmetic above, 320 at five instead of three waves per
// SIMD, 261 with the query form.

// DPP move inside a quad
template <int CTRL>
__device__ __forceinline__ uint32_t qdpp(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, true);
}
template <int CTRL>
__device__ __forceinline__ float qdppf(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}

// RegionNeighbours<8>::sampleApproximateClosestRegionIdx (spatial/KNN.h:134-148)
// on a quad: lane q holds the keys of slots q and q + 4 (squared distance with
// the slot in the low 3 bits, +inf for empty slots; keys are distinct, and as
// unsigned integers in the order of the floats), ranks them among the eight,
// and the slot of rank `sel` is the pick.
__device__ __forceinline__ uint32_t quad_knn_pick(const QueryField& f, uint32_t leaf, int q, float x, float y, float z,
                                                  float* u) {
  const uint32_t sel = knn_draw(u, f.nbSize);
  uint32_t id[2], key[2];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const uint32_t s = (uint32_t)(q + 4 * h);
    id[h] = f.nbIds[leaf * 8 + s];
    const float4 p = f.nbPts[leaf * 8 + s];
    const float d = knn_d2(p.x - x, p.y - y, p.z - z, f.knnFused != 0);
    key[h] = ((id[h] == 0xffffffffu ? 0x7f800000u : __float_as_uint(d)) & ~7u) | s;
  }
  uint32_t rank[2] = {key[1] < key[0] ? 1u : 0u, key[0] < key[1] ? 1u : 0u};
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const uint32_t a = qdpp<0xB1>(key[h]), b = qdpp<0x4E>(key[h]), c = qdpp<0x1B>(key[h]);  // lanes q ^ 1, 2, 3
#pragma unroll
    for (int g = 0; g < 2; g++)
      rank[g] += (a < key[g] ? 1u : 0u) + (b < key[g] ? 1u : 0u) + (c < key[g] ? 1u : 0u);
  }
  uint32_t r = (rank[0] == sel ? id[0] : 0u) | (rank[1] == sel ? id[1] : 0u);
  r |= qdpp<0xB1>(r);
  r |= qdpp<0x4E>(r);
  return r;
}

__device__ __forceinline__ int lookup_region(const QueryField& f, int q, float x, float y, float z, float* u,
                                             uint32_t& id) {
  if (!f.trained) return -1;
  if (!(x >= f.lo[0] && x <= f.hi[0] && y >= f.lo[1] && y <= f.hi[1] && z >= f.lo[2] && z <= f.hi[2])) return -1;
  uint32_t i = 0;
  KDNode nd = f.nodes[0];
  while (!nd.isLeaf()) {
    const uint32_t d = nd.dim();
    const float p = d == 0 ? x : (d == 1 ? y : z);
    i = nd.idx() + (p >= nd.pivot ? 1u : 0u);
    nd = f.nodes[i];
  }
  const uint32_t leaf = nd.idx();
  id = leaf;
  if (f.knn && *u >= 0.f) return (int)quad_knn_pick(f, leaf, q, x, y, z, u);
  return (int)leaf;
}

// sum over the quad; the same bits in its four lanes (IEEE addition commutes)
__device__ __forceinline__ float qsum4(float v) {
  v += qdppf<0xB1>(v);  // lanes q ^ 1
  v += qdppf<0x4E>(v);  // lanes q ^ 2
  return v;
}

// value of quad lane 0, 1, 2 or 3 (DPP quad broadcast)
template <int L>
__device__ __forceinline__ float qlane(float v) {
  return qdppf<L * 0x55>(v);
}

// Correctly rounded n / d by the steps of the compiler's division (one
// refinement of the reciprocal, two of the quotient), the reciprocal formed
// once per d, without the scaling that only operands near the ends of the
// exponent range need: the same quotient while d, n and n / d lie within
// 2^-100 .. 2^100 (or n is 0).  A smaller n, whose remainders are rounded to
// denormals, may end a unit in the last place off: a coordinate under 2^-50 of
// its vector's length, or a component's share under 2^-33 of the integral.
struct Recip {
  float d, r;
};
__device__ __forceinline__ Recip recip_of(float d) {
  const float r = __builtin_amdgcn_rcpf(d);
  return {d, fmaf(fmaf(-d, r, 1.f), r, r)};
}
__device__ __forceinline__ float div_by(float n, const Recip& k) {
  float q = n * k.r;
  q = fmaf(fmaf(-k.d, q, n), k.r, q);
  return fmaf(fmaf(-k.d, q, n), k.r, q);
}

// correctly rounded square root (x within 2^-90 .. 2^120, or 0): the nearest
// of the hardware's estimate and its two neighbours
__device__ __forceinline__ float sqrt_in_range(float x) {
  const float s = __builtin_amdgcn_sqrtf(x);
  const float dn = __int_as_float(__float_as_int(s) - 1), up = __int_as_float(__float_as_int(s) + 1);
  const float ed = fmaf(-dn, s, x), eu = fmaf(-up, s, x);
  const float r = ed <= 0.f ? dn : s;
  return eu > 0.f ? up : r;
}

// This lane's components (k = 4j + q) after the parallax shift to the query
// position: their directions, formed once per query and shared by every
// product below.  Slots from K on hold a zero-weight component.
struct LaneShift {
  float mx[8], my[8], mz[8];
};

// A region's components as 16-byte halves: direction and distance, then weight,
// concentration and normalisation (RegionState::QueryComp).
struct Mixture {
  const float4* q;
  int K;
  __device__ __forceinline__ float4 dir(int k) const { return q[2 * k]; }
  __device__ __forceinline__ float4 lobe(int k) const { return q[2 * k + 1]; }
};

__device__ __forceinline__ void lane_shift(const Mixture& V, int k, bool par, float sx, float sy, float sz, float& mx,
                                           float& my, float& mz) {
  const float4 a = V.dir(k);
  mx = a.x;
  my = a.y;
  mz = a.z;
  if (par) {  // shift_comp
    const float d = a.w;
    const float px = fmaf(mx, d, sx), py = fmaf(my, d, sy), pz = fmaf(mz, d, sz);
    const float l = sqrt_in_range(qdot(px, py, pz, px, py, pz));
    const Recip rl = recip_of(l);
    float qx = div_by(px, rl), qy = div_by(py, rl), qz = div_by(pz, rl);
    // a length out of the root's or the quotients' range (a component may carry
    // any distance): the scaled forms, which give the other lanes the same bits
    if (__ballot(!(l > 1e-13f && l < 1e18f)) != 0) {
      const float ls = sqrtf(qdot(px, py, pz, px, py, pz));
      qx = px / ls;
      qy = py / ls;
      qz = pz / ls;
    }
    const bool shift = d > 0.f && isfinite(d);  // (formed before the divisions: 277 instead of 261 us, above)
    mx = shift ? qx : mx;
    my = shift ? qy : my;
    mz = shift ? qz : mz;
  }
}

// Product of one shifted component with the lobe (weight, n, kn, nn):
// product_comp of query_math.h with shared reciprocals and every fused
// multiply-add written out (each use of it rounds alike).
__device__ __forceinline__ ProdComp lane_product(const float4 b, float mx, float my, float mz, float weight,
                                                 float nx, float ny, float nz, float kn, float nn) {
  const float w = b.x, kappa = b.y, norm = b.z;
  ProdComp p;
  float ax = fmaf(kappa, mx, kn * nx), ay = fmaf(kappa, my, kn * ny), az = fmaf(kappa, mz, kn * nz);
  float nk = sqrt_in_range(qdot(ax, ay, az, ax, ay, az));
  const bool ok = nk > 1e-3f;
  nk = ok ? nk : 0.f;
  const Recip k = recip_of(nk);
  ax = ok ? div_by(ax, k) : mx;
  ay = ok ? div_by(ay, k) : my;
  az = ok ? div_by(az, k) : mz;
  const float e = expf(-2.f * nk);
  float nrm = div_by(nk, recip_of(2.f * 3.14159265358979f * (1.f - e)));
  nrm = ok ? nrm : kOneOverFourPi;
  float scale = div_by(norm * nn, recip_of(nrm));
  const float c0 = qdot(mx, my, mz, ax, ay, az);
  const float c1 = qdot(nx, ny, nz, ax, ay, az);
  scale *= expf(fmaf(kappa, c0 - 1.f, kn * (c1 - 1.f)));
  scale *= w * weight;
  p.scale = scale;
  p.kappa = nk;
  p.mx = ax;
  p.my = ay;
  p.mz = az;
  p.norm = nrm;
  p.em2k = e;
  return p;
}

// part + eval_comp(...)
__device__ __forceinline__ float eval_add(float part, float w, float norm, float kappa, float mx, float my, float mz,
                                          float dx, float dy, float dz) {
  const float c = qdot(dx, dy, dz, mx, my, mz);
  return fmaf(norm * expf(kappa * fminf(c - 1.f, 0.f)), w, part);
}

// Calls f(j) for the component groups j < J (J uniform over the wave), two
// groups per branch.
template <class F>
__device__ __forceinline__ void for_groups(int J, F&& f) {
#pragma unroll
  for (int j = 0; j < 8; j += 2) {
    if (j < J) {
      f(j);
      f(j + 1);
    }
  }
}

// Products of this lane's shifted components with the cosine lobe, held from
// the integral to the pdf: scale 0 for k >= K.
struct LaneComps {
  float s[8], kap[8], mx[8], my[8], mz[8], nrm[8];
};

// pdf at direction d of the product held in c (quad sum)
__device__ __forceinline__ float quad_pdf(const Mixture& V, int q, int J, const LaneComps& c, float integral,
                                          float dx, float dy, float dz) {
  const float inv = 1.f / integral;
  const int K = V.K;
  float part = 0.f;
  for_groups(J, [&](int j) {
    const float v = eval_add(part, c.s[j] * inv, c.nrm[j], c.kap[j], c.mx[j], c.my[j], c.mz[j], dx, dy, dz);
    part = 4 * j + q < K ? v : part;
  });
  return qsum4(part);
}

// pdf at d of the product with a lobe, the products formed on the fly (quad sum)
__device__ __forceinline__ float quad_pdf_lobe(const Mixture& V, int q, int J, const LaneShift& h, float weight,
                                               float nx, float ny, float nz, float kn, float nn, float integral,
                                               float dx, float dy, float dz) {
  const float inv = 1.f / integral;
  const int K = V.K;
  float part = 0.f;
  for_groups(J, [&](int j) {
    const int k = 4 * j + q;
    const ProdComp p =
        lane_product(V.lobe(k), h.mx[j], h.my[j], h.mz[j], weight, nx, ny, nz, kn, nn);
    const float v = eval_add(part, p.scale * inv, p.norm, p.kappa, p.mx, p.my, p.mz, dx, dy, dz);
    part = k < K ? v : part;
  });
  return qsum4(part);
}

// sum of this lane's product weights over the quad
__device__ __forceinline__ float quad_integral(const float s[8]) {
  float part = 0.f;
#pragma unroll
  for (int j = 0; j < 8; j++) part += s[j];
  return qsum4(part);
}

// The component PAVMM::sample takes for u1: the first k, in component order,
// whose cumulative share of the integral reaches u1 (the last one if rounding
// leaves the total short).  The walk goes over groups of four components (one
// per lane; `group(j)` is called for every group until it is found, with
// whether it is the one) and then inside the chosen group.  u1 is rescaled to
// the component's share.
struct Pick {
  int js, qs;  // component 4 js + qs
  float us;
};
template <class F>
__device__ __forceinline__ Pick quad_pick(const Mixture& V, int Jw, const float s[8], float integral, float u1,
                                          F&& group) {
  const int K = V.K;
  const int J = (K + 3) >> 2;
  // an integral near the ends of the exponent range needs the scaled division
  const bool plain = __ballot(!(integral > 1e-20f && integral < 1e20f)) == 0;
  const Recip ri = recip_of(integral);
  float acc = 0.f, accs = 0.f;  // share of the groups before the chosen one
  float x = 0.f;                // this lane's share in the chosen group
  int js = -1;
  for_groups(Jw, [&](int j) {
    float sh = div_by(s[j], ri);
    if (!plain) sh = s[j] / integral;
    const float g = qsum4(sh);
    const bool open = js < 0 && j < J;
    const bool take = open && (acc + g >= u1 || j == J - 1);  // the last group is walked in any case
    js = take ? j : js;
    accs = take ? acc : accs;
    x = take ? sh : x;
    group(j, take);
    acc = open ? acc + g : acc;
  });
  const float x0 = qlane<0>(x), x1 = qlane<1>(x), x2 = qlane<2>(x), x3 = qlane<3>(x);
  const int last = 4 * js + 3 < K ? 3 : ((K - 1) & 3);  // last component of the group
  // the walk inside the group: components 4 js + l, l = 0 .. last
  float sum = accs;
  int qs = last;
  if (last > 0 && sum + x0 >= u1) qs = 0;
  else {
    if (last > 0) sum += x0;
    if (last > 1 && sum + x1 >= u1) qs = 1;
    else {
      if (last > 1) sum += x1;
      if (last > 2 && sum + x2 >= u1) qs = 2;
      else if (last > 2) sum += x2;
    }
  }
  const float cdf = qs == 0 ? x0 : (qs == 1 ? x1 : (qs == 2 ? x2 : x3));
  return {js, qs, fminf(1.f - 1.19209290e-7f, (u1 - sum) / cdf)};
}

// largest component group count of the wave's active lanes
__device__ __forceinline__ int wave_groups(int K) {
  int J = 8;
  while (J > 1 && __ballot(K > 4 * (J - 1)) == 0) J--;
  return J;
}

// One query on the four lanes of a quad: lookup (+ KNN pick), parallax shift,
// cosine (surface) or 3-lobe HG (volume) product, one sample and its pdf.
// Invalid queries (outside the field, untrained field, invalid region) give
// dir 0, pdf 0, id ~0.  Every lane returns the same results.  VOLUMES: the
// batch may hold volume queries (their registers are most of the kernel's: a
// batch of surface queries alone runs five waves to a SIMD, with them four).
template <bool VOLUMES>
__device__ __forceinline__ void query_quad(const QueryField& surf, const QueryField& vol, const HGRep* __restrict__ hg,
                                           bool volume, float x, float y, float z, float nx, float ny, float nz,
                                           float g, float ux, float uy, float u, float out[3], float& pdf,
                                           uint32_t& id, float& integral) {
  const QueryField& f = VOLUMES && volume ? vol : surf;
  const int lane = threadIdx.x & 63, q = lane & 3;
  id = 0xffffffffu;
  pdf = 0.f;
  integral = 0.f;
  out[0] = out[1] = out[2] = 0.f;
  const int r = lookup_region(f, q, x, y, z, &u, id);
  if (r < 0 || !f.regions[r].valid) {
    id = 0xffffffffu;
    return;
  }
  const RegionState& S = f.regions[r];
  const Mixture V{(const float4*)S.query, S.vmm.K};
  const bool par = f.parallax != 0;
  const float sx = S.vmm.pivot[0] - x, sy = S.vmm.pivot[1] - y, sz = S.vmm.pivot[2] - z;
  const int K = V.K;
  const int J = wave_groups(K);
  if (!VOLUMES || !volume) {
    const float kn = kCosineKappa, nn = cosine_normalization();
    LaneComps c;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      c.s[j] = 0.f; c.kap[j] = 0.f; c.mx[j] = 0.f; c.my[j] = 0.f; c.mz[j] = 1.f; c.nrm[j] = 0.f;
    }
    for_groups(J, [&](int j) {
      const int k = 4 * j + q;
      float hx, hy, hz;
      lane_shift(V, k, par, sx, sy, sz, hx, hy, hz);
      const ProdComp p = lane_product(V.lobe(k), hx, hy, hz, 1.f, nx, ny, nz, kn, nn);
      c.s[j] = k < K ? p.scale : 0.f; c.kap[j] = p.kappa; c.mx[j] = p.mx; c.my[j] = p.my; c.mz[j] = p.mz;
      c.nrm[j] = p.norm;
    });
    integral = quad_integral(c.s);
    float kap = 0.f, mx = 0.f, my = 0.f, mz = 1.f;  // of this lane's component in the chosen group
    const Pick pk = quad_pick(V, J, c.s, integral, uy, [&](int j, bool take) {
      kap = take ? c.kap[j] : kap;
      mx = take ? c.mx[j] : mx;
      my = take ? c.my[j] : my;
      mz = take ? c.mz[j] : mz;
    });
    const int src = (lane & ~3) | pk.qs;
    kap = __shfl(kap, src);
    sample_comp(kap, expf(-2.f * kap), __shfl(mx, src), __shfl(my, src), __shfl(mz, src), ux, pk.us, out);
    pdf = quad_pdf(V, q, J, c, integral, out[0], out[1], out[2]);
  } else {
    const HGRep& rep = hg[hg_index(g)];
    const int KP = (int)rep.K;
    LaneShift h;
    for_groups(J, [&](int j) { lane_shift(V, 4 * j + q, par, sx, sy, sz, h.mx[j], h.my[j], h.mz[j]); });
    // the product weights of every lobe are kept; of the products themselves
    // only the sampled component's is formed again
    float s[4][8], integ[4], mw[4], sgn[4];
    float sum = 0.f;
#pragma unroll
    for (int m = 0; m < 4; m++) {
#pragma unroll
      for (int j = 0; j < 8; j++) s[m][j] = 0.f;
      integ[m] = 0.f;
      sgn[m] = 1.f;
      if (__ballot(m < KP) != 0) {
        sgn[m] = (g * rep.mc[m] > 0.f) ? 1.f : -1.f;
        const float weight = rep.w[m], kn = rep.kappa[m], nn = rep.norm[m];
        for_groups(J, [&](int j) {
          const int k = 4 * j + q;
          const ProdComp p = lane_product(V.lobe(k), h.mx[j], h.my[j], h.mz[j], weight,
                                          nx * sgn[m], ny * sgn[m], nz * sgn[m], kn, nn);
          s[m][j] = k < K ? p.scale : 0.f;
        });
        integ[m] = quad_integral(s[m]);
        sum = m < KP ? sum + integ[m] : sum;
      }
    }
#pragma unroll
    for (int m = 0; m < 4; m++) mw[m] = integ[m] / sum;
    // the lobe: the first whose cumulative share exceeds ux (the last one in any case)
    float acc = 0.f;
    int lobe = 0;
    bool open = true;
#pragma unroll
    for (int m = 0; m < 3; m++) {
      const float nw = acc + mw[m];
      open = open && m < KP - 1 && !(nw > ux);
      acc = open ? nw : acc;
      lobe = open ? m + 1 : lobe;
    }
    float sl[8], integral1 = integ[0], w1 = mw[0], sg = sgn[0];
#pragma unroll
    for (int j = 0; j < 8; j++) sl[j] = s[0][j];
#pragma unroll
    for (int m = 1; m < 4; m++) {
      const bool it = lobe == m;
      integral1 = it ? integ[m] : integral1;
      w1 = it ? mw[m] : w1;
      sg = it ? sgn[m] : sg;
#pragma unroll
      for (int j = 0; j < 8; j++) sl[j] = it ? s[m][j] : sl[j];
    }
    const Pick pk = quad_pick(V, J, sl, integral1, uy, [](int, bool) {});
    const int k = 4 * pk.js + pk.qs;
    float hx, hy, hz;
    lane_shift(V, k, par, sx, sy, sz, hx, hy, hz);
    const ProdComp p = lane_product(V.lobe(k), hx, hy, hz, rep.w[lobe], nx * sg, ny * sg, nz * sg,
                                    rep.kappa[lobe], rep.norm[lobe]);
    sample_comp(p.kappa, p.em2k, p.mx, p.my, p.mz, (ux - acc) / w1, pk.us, out);
#pragma unroll
    for (int m = 0; m < 4; m++) {
      if (__ballot(m < KP) == 0) continue;
      const float v = quad_pdf_lobe(V, q, J, h, rep.w[m], nx * sgn[m], ny * sgn[m], nz * sgn[m], rep.kappa[m],
                                    rep.norm[m], integ[m], out[0], out[1], out[2]);
      pdf = m < KP ? fmaf(mw[m], v, pdf) : pdf;
    }
    integral = sum;
  }
}

template <bool VOLUMES>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(VOLUMES ? 4 : 5))) k_query(QueryField surf, QueryField vol, const HGRep* __restrict__ hg,
                                               uint32_t n, const float* __restrict__ pos, const float* __restrict__ nrm,
                                               const float* __restrict__ gArr, const float* __restrict__ u2,
                                               const float* __restrict__ u1, const uint8_t* __restrict__ isVolume,
                                               float* __restrict__ dirOut, float* __restrict__ pdfOut,
                                               uint32_t* __restrict__ idOut, float* __restrict__ integralOut) {
  const uint32_t i = (uint32_t)(((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 2);  // this quad's query
  if (i >= n) return;
  const bool volume = isVolume ? isVolume[i] != 0 : false;
  float out[3], pdf, integral;
  uint32_t id;
  query_quad<VOLUMES>(surf, vol, hg, volume, pos[3 * i], pos[3 * i + 1], pos[3 * i + 2], nrm[3 * i], nrm[3 * i + 1],
             nrm[3 * i + 2], gArr ? gArr[i] : 0.f, u2[2 * i], u2[2 * i + 1], u1 ? u1[i] : -1.f, out, pdf, id, integral);
  if ((threadIdx.x & 3) != 0) return;
  dirOut[3 * i] = out[0];
  dirOut[3 * i + 1] = out[1];
  dirOut[3 * i + 2] = out[2];
  pdfOut[i] = pdf;
  if (idOut) idOut[i] = id;
  if (integralOut) integralOut[i] = integral;
}

// Batch of pieces: the quad of query i of the batch finds its piece (pieces
// ordered by begin) and works on query i - begin of it through the piece's
// pointers.
template <bool VOLUMES>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(VOLUMES ? 4 : 5))) k_query_pieces(QueryField surf, QueryField vol, const HGRep* __restrict__ hg,
                                                      const QueryPiece* __restrict__ pieces, uint32_t numPieces,
                                                      uint32_t n) {
  const uint32_t i = (uint32_t)(((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 2);
  if (i >= n) return;
  uint32_t lo = 0, hi = numPieces;  // last piece with begin <= i
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (pieces[mid].begin <= i) lo = mid; else hi = mid;
  }
  const QueryPiece& P = pieces[lo];
  const uint32_t j = i - P.begin;
  if (j >= P.n) return;
  const bool volume = P.vol ? P.vol[j] != 0 : false;
  float out[3], pdf, integral;
  uint32_t id;
  query_quad<VOLUMES>(surf, vol, hg, volume, P.pos[3 * j], P.pos[3 * j + 1], P.pos[3 * j + 2], P.nrm[3 * j], P.nrm[3 * j + 1],
             P.nrm[3 * j + 2], P.g ? P.g[j] : 0.f, P.u2[2 * j], P.u2[2 * j + 1], P.u1 ? P.u1[j] : -1.f, out, pdf, id,
             integral);
  if ((threadIdx.x & 3) != 0) return;
  P.dir[3 * j] = out[0];
  P.dir[3 * j + 1] = out[1];
  P.dir[3 * j + 2] = out[2];
  P.pdf[j] = pdf;
  if (P.id) P.id[j] = id;
  if (P.integral) P.integral[j] = integral;
}

void launch_query_pieces(const QueryField& surf, const QueryField& vol, const HGRep* hg, const QueryPiece* pieces,
                         uint32_t numPieces, uint32_t n, bool volumes, hipStream_t s) {
  if (n == 0 || numPieces == 0) return;
  hipLaunchKernelGGL(volumes ? k_query_pieces<true> : k_query_pieces<false>, dim3((n + 63) / 64), dim3(256), 0, s, surf, vol, hg, pieces, numPieces, n);
}

void launch_query(const QueryField& surf, const QueryField& vol, const HGRep* hg, uint32_t n, const float* pos,
                  const float* nrm, const float* g, const float* u2, const float* u1, const uint8_t* isVolume,
                  float* dirOut, float* pdfOut, uint32_t* idOut, float* integralOut, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(isVolume ? k_query<true> : k_query<false>, dim3((n + 63) / 64), dim3(256), 0, s, surf, vol, hg, n,
                     pos, nrm, g, u2, u1, isVolume, dirOut, pdfOut, idOut, integralOut);
}

}  // namespace pglgpu
