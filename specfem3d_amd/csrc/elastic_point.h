// elastic_point.h -- per-GLL-point arithmetic of the isotropic elastic stiffness, shared by the
// single-shot point-per-lane kernel (k_elastic.hip) and the batched many-shot kernel
// (k_batch.hip). Every expression keeps the reference's operand order
// (compute_forces_viscoelastic.F90:331-335 contractions, :420-461 mapping, :616-630 stress,
// :661-710 test-function products, :722-726 divergence, :788-806 weights), so the exact build
// (-ffp-contract=off) reproduces the CPU solver bit for bit whichever kernel runs it.
//
// Element tiles live in LDS with the value of point q = i + 5 j + 25 k at base[q * PS]: PS = 1 for
// one field per workgroup, PS = shots per workgroup for shot-interleaved tiles. The GLL tables
// (hp[i*5+l] = hprime, hpw[i*5+l] = hprimewgll, wxy[a*5+b] = wgllwgll) are read through pointers:
// the kernels stage them in LDS so a lane reads each coefficient when it uses it instead of
// holding its 33 coefficients in registers.
#pragma once

#include "kernels.h"

#ifndef SF_EXACT
#define SF_EXACT 1
#endif
// FMA builds fold, on regular elements, xix_regular into hprime and jacobian_regular *
// xix_regular into hprimewgll (the tables at sG + 75 and sG + 100): the nine-term mapping of the
// gradient and the eighteen multiplies of the test-function products become copies. The exact
// builds keep the reference's operation order.
#define SF_FOLD (!SF_EXACT)

namespace sf {

// Workgroup barrier that orders LDS accesses only: this wave's LDS operations complete
// (lgkmcnt(0)), then s_barrier; the "memory" clobber keeps the compiler from moving memory
// accesses across it. Global loads, stores and atomics issued earlier, and LDS-direct loads
// (global_load_lds, which complete through vmcnt and are read back only by the lane that issued
// them), stay in flight across it; __syncthreads would wait for all of them (vmcnt(0)).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

struct Grad9 {  // d/dxi, d/deta, d/dgamma of the three components
  realw x1, y1, z1, x2, y2, z2, x3, y3, z3;
};

struct JacPt {  // inverse-Jacobian terms and determinant at one point (irregular elements)
  realw xix, xiy, xiz, etax, etay, etaz, gax, gay, gaz, jac;
};

// Sums of products, left to right. FMA builds name the one product that is rounded by itself, the second: which
// one the compiler takes depends on the code around it, and records of a weak first arrival show the
// difference (their largest part is what rounding leaves behind the front).
__device__ __forceinline__ realw add_product(realw sum, realw a, realw b) {
#if SF_EXACT
  return sum + a * b;
#else
  return fmaf(a, b, sum);
#endif
}
__device__ __forceinline__ realw sum2(realw a1, realw b1, realw a2, realw b2) {
#if SF_EXACT
  return a1 * b1 + a2 * b2;
#else
  return fmaf(a1, b1, a2 * b2);
#endif
}
__device__ __forceinline__ realw sum3(realw a1, realw b1, realw a2, realw b2, realw a3, realw b3) {
  return add_product(sum2(a1, b1, a2, b2), a3, b3);
}

// tempx1 = sum_l hprime(i,l) u(l,j,k), tempx2 = sum_l hprime(j,l) u(i,l,k),
// tempx3 = sum_l hprime(k,l) u(i,j,l), summed left to right.
template <int PS>
__device__ __forceinline__ Grad9 tile_gradient(const realw* sx, const realw* sy, const realw* sz, const realw* hp,
                                               int i, int j, int k) {
  const int b1 = 5 * j + 25 * k, b2 = i + 25 * k, b3 = i + 5 * j;
  Grad9 t;
  {
    const realw h1 = hp[i * 5], h2 = hp[j * 5], h3 = hp[k * 5];
    const realw a1 = hp[i * 5 + 1], a2 = hp[j * 5 + 1], a3 = hp[k * 5 + 1];
    const int p1 = b1 * PS, p2 = b2 * PS, p3 = b3 * PS, q1 = (b1 + 1) * PS, q2 = (b2 + 5) * PS, q3 = (b3 + 25) * PS;
    t.x1 = sum2(h1, sx[p1], a1, sx[q1]); t.y1 = sum2(h1, sy[p1], a1, sy[q1]); t.z1 = sum2(h1, sz[p1], a1, sz[q1]);
    t.x2 = sum2(h2, sx[p2], a2, sx[q2]); t.y2 = sum2(h2, sy[p2], a2, sy[q2]); t.z2 = sum2(h2, sz[p2], a2, sz[q2]);
    t.x3 = sum2(h3, sx[p3], a3, sx[q3]); t.y3 = sum2(h3, sy[p3], a3, sy[q3]); t.z3 = sum2(h3, sz[p3], a3, sz[q3]);
  }
#pragma unroll
  for (int l = 2; l < 5; l++) {
    const realw a1 = hp[i * 5 + l], a2 = hp[j * 5 + l], a3 = hp[k * 5 + l];
    const int q1 = (b1 + l) * PS, q2 = (b2 + 5 * l) * PS, q3 = (b3 + 25 * l) * PS;
    t.x1 = add_product(t.x1, a1, sx[q1]); t.y1 = add_product(t.y1, a1, sy[q1]); t.z1 = add_product(t.z1, a1, sz[q1]);
    t.x2 = add_product(t.x2, a2, sx[q2]); t.y2 = add_product(t.y2, a2, sy[q2]); t.z2 = add_product(t.z2, a2, sz[q2]);
    t.x3 = add_product(t.x3, a3, sx[q3]); t.y3 = add_product(t.y3, a3, sy[q3]); t.z3 = add_product(t.z3, a3, sz[q3]);
  }
  return t;
}

// Strain at u + dt v (attenuation, compute_forces_viscoelastic.F90:396-417): each contraction of u
// is continued with the five terms of the dt*v tile.
template <int PS>
__device__ __forceinline__ Grad9 tile_gradient_continue(Grad9 t, const realw* wx, const realw* wy, const realw* wz,
                                                        const realw* hp, int i, int j, int k) {
  const int b1 = 5 * j + 25 * k, b2 = i + 25 * k, b3 = i + 5 * j;
#pragma unroll
  for (int l = 0; l < 5; l++) {
    const realw h1 = hp[i * 5 + l], h2 = hp[j * 5 + l], h3 = hp[k * 5 + l];
    const int q1 = (b1 + l) * PS, q2 = (b2 + 5 * l) * PS, q3 = (b3 + 25 * l) * PS;
    t.x1 = add_product(t.x1, wx[q1], h1); t.y1 = add_product(t.y1, wy[q1], h1); t.z1 = add_product(t.z1, wz[q1], h1);
    t.x2 = add_product(t.x2, wx[q2], h2); t.y2 = add_product(t.y2, wy[q2], h2); t.z2 = add_product(t.z2, wz[q2], h2);
    t.x3 = add_product(t.x3, wx[q3], h3); t.y3 = add_product(t.y3, wy[q3], h3); t.z3 = add_product(t.z3, wz[q3], h3);
  }
  return t;
}

// The nine displacement derivatives in (x, y, z): d(ux)/dx .. d(uz)/dz.
struct Du9 {
  realw xx, xy, xz, yx, yy, yz, zx, zy, zz;
};

template <bool FOLD = SF_FOLD>
__device__ __forceinline__ Du9 map_gradient(const Grad9& t, bool irr, const JacPt& J, realw xr) {
  Du9 d;
  if (irr) {
    d.xx = sum3(J.xix, t.x1, J.etax, t.x2, J.gax, t.x3);
    d.xy = sum3(J.xiy, t.x1, J.etay, t.x2, J.gay, t.x3);
    d.xz = sum3(J.xiz, t.x1, J.etaz, t.x2, J.gaz, t.x3);
    d.yx = sum3(J.xix, t.y1, J.etax, t.y2, J.gax, t.y3);
    d.yy = sum3(J.xiy, t.y1, J.etay, t.y2, J.gay, t.y3);
    d.yz = sum3(J.xiz, t.y1, J.etaz, t.y2, J.gaz, t.y3);
    d.zx = sum3(J.xix, t.z1, J.etax, t.z2, J.gax, t.z3);
    d.zy = sum3(J.xiy, t.z1, J.etay, t.z2, J.gay, t.z3);
    d.zz = sum3(J.xiz, t.z1, J.etaz, t.z2, J.gaz, t.z3);
  } else if (FOLD) {
    d.xx = t.x1; d.xy = t.x2; d.xz = t.x3;
    d.yx = t.y1; d.yy = t.y2; d.yz = t.y3;
    d.zx = t.z1; d.zy = t.z2; d.zz = t.z3;
  } else {
    d.xx = xr * t.x1; d.xy = xr * t.x2; d.xz = xr * t.x3;
    d.yx = xr * t.y1; d.yy = xr * t.y2; d.yz = xr * t.y3;
    d.zx = xr * t.z1; d.zy = xr * t.z2; d.zz = xr * t.z3;
  }
  return d;
}

struct Sigma6 {
  realw xx, yy, zz, xy, xz, yz;
};

// isotropic stress, lambda + 2 mu = kappa + 4/3 mu, lambda = (lambda + 2 mu) - 2 mu
__device__ __forceinline__ Sigma6 iso_stress(const Du9& d, realw kappal, realw mul) {
  const realw FOUR_THIRDS = (realw)4 / (realw)3;
  const realw lp2m = kappal + FOUR_THIRDS * mul;
  const realw lambdal = lp2m - (realw)2 * mul;
  Sigma6 s;
#if SF_EXACT
  s.xx = lp2m * d.xx + lambdal * (d.yy + d.zz);
  s.yy = lp2m * d.yy + lambdal * (d.xx + d.zz);
  s.zz = lp2m * d.zz + lambdal * (d.xx + d.yy);
#else
  s.xx = fmaf(lp2m, d.xx, lambdal * (d.yy + d.zz));
  s.yy = fmaf(lp2m, d.yy, lambdal * (d.xx + d.zz));
  s.zz = fmaf(lambdal, d.xx + d.yy, lp2m * d.zz);  // the other product here: as it has always been rounded
#endif
  s.xy = mul * (d.xy + d.yx);
  s.xz = mul * (d.zx + d.xz);
  s.yz = mul * (d.zy + d.yz);
  return s;
}

// jacobian * sigma . (dxi/dx), (deta/dx), (dgamma/dx): t[0..2] xi, t[3..5] eta, t[6..8] gamma
// (VISCO: the kernels with memory variables, whose FMA builds round another of the products by itself)
template <bool FOLD = SF_FOLD, bool VISCO = false>
__device__ __forceinline__ void stress_products(const Sigma6& s, bool irr, const JacPt& J, realw jacl, realw xr,
                                                realw t[9]) {
  const realw syx = s.xy, szx = s.xz, szy = s.yz;
  if (irr) {
    t[0] = jacl * (VISCO ? sum3(s.xx, J.xix, syx, J.xiy, szx, J.xiz) : sum3(syx, J.xiy, s.xx, J.xix, szx, J.xiz));
    t[1] = jacl * (VISCO ? sum3(s.yy, J.xiy, s.xy, J.xix, szy, J.xiz) : sum3(s.xy, J.xix, s.yy, J.xiy, szy, J.xiz));
    t[2] = jacl * sum3(s.xz, J.xix, s.yz, J.xiy, s.zz, J.xiz);
    t[3] = jacl * (VISCO ? sum3(s.xx, J.etax, syx, J.etay, szx, J.etaz) : sum3(syx, J.etay, s.xx, J.etax, szx, J.etaz));
    t[4] = jacl * (VISCO ? sum3(s.yy, J.etay, s.xy, J.etax, szy, J.etaz) : sum3(s.xy, J.etax, s.yy, J.etay, szy, J.etaz));
    t[5] = jacl * sum3(s.xz, J.etax, s.yz, J.etay, s.zz, J.etaz);
    t[6] = jacl * (VISCO ? sum3(s.xx, J.gax, syx, J.gay, szx, J.gaz) : sum3(syx, J.gay, s.xx, J.gax, szx, J.gaz));
    t[7] = jacl * (VISCO ? sum3(s.yy, J.gay, s.xy, J.gax, szy, J.gaz) : sum3(s.xy, J.gax, s.yy, J.gay, szy, J.gaz));
    t[8] = jacl * sum3(s.xz, J.gax, s.yz, J.gay, s.zz, J.gaz);
  } else if (FOLD) {
    t[0] = s.xx; t[1] = s.xy; t[2] = s.xz;
    t[3] = syx;  t[4] = s.yy; t[5] = s.yz;
    t[6] = szx;  t[7] = szy;  t[8] = s.zz;
  } else {
    t[0] = jacl * s.xx * xr;
    t[1] = jacl * s.xy * xr;
    t[2] = jacl * s.xz * xr;
    t[3] = jacl * syx * xr;
    t[4] = jacl * s.yy * xr;
    t[5] = jacl * s.yz * xr;
    t[6] = jacl * szx * xr;
    t[7] = jacl * szy * xr;
    t[8] = jacl * s.zz * xr;
  }
}

// f_c = wgllwgll_yz(j,k) sum_l hprimewgll(l,i) t1_c(l,j,k) + wgllwgll_xz(i,k) sum_l hprimewgll(l,j) t2_c(i,l,k)
//     + wgllwgll_xy(i,j) sum_l hprimewgll(l,k) t3_c(i,j,l); plane m of the tile at sT + m * plane.
template <int PS>
__device__ __forceinline__ realw tile_divergence_c(const realw* sT, int plane, const realw* hpw, const realw* wxy,
                                                   int i, int j, int k, int cc) {
  const int b1 = 5 * j + 25 * k, b2 = i + 25 * k, b3 = i + 5 * j;
  const realw *s1 = sT + cc * plane, *s2 = sT + (3 + cc) * plane, *s3 = sT + (6 + cc) * plane;
  realw n1 = sum2(hpw[i], s1[b1 * PS], hpw[5 + i], s1[(b1 + 1) * PS]);
  realw n2 = sum2(hpw[j], s2[b2 * PS], hpw[5 + j], s2[(b2 + 5) * PS]);
  realw n3 = sum2(hpw[k], s3[b3 * PS], hpw[5 + k], s3[(b3 + 25) * PS]);
#pragma unroll
  for (int l = 2; l < 5; l++) {
    n1 = add_product(n1, hpw[l * 5 + i], s1[(b1 + l) * PS]);
    n2 = add_product(n2, hpw[l * 5 + j], s2[(b2 + 5 * l) * PS]);
    n3 = add_product(n3, hpw[l * 5 + k], s3[(b3 + 25 * l) * PS]);
  }
  return sum3(wxy[j * 5 + k], n1, wxy[i * 5 + k], n2, wxy[i * 5 + j], n3);
}
template <int PS>
__device__ __forceinline__ void tile_divergence(const realw* sT, int plane, const realw* hpw, const realw* wxy, int i,
                                                int j, int k, realw f[3]) {
#pragma unroll
  for (int cc = 0; cc < 3; cc++) f[cc] = tile_divergence_c<PS>(sT, plane, hpw, wxy, i, j, k, cc);
}

// stage the GLL coefficients of G in LDS (lanes 0..124 of the workgroup; needs a barrier before
// use): hp, hpw, wxy, and the folded hpr, hpwr at sG + 75, sG + 100
constexpr int SF_NGLL_TABLE = 125;
__device__ __forceinline__ void stage_gll(realw* sG, const GLLk& G, int lane) {
  if (lane < 25) sG[lane] = G.hp[lane];
  else if (lane < 50) sG[lane] = G.hpw[lane - 25];
  else if (lane < 75) sG[lane] = G.wxy[lane - 50];
  else if (lane < 100) sG[lane] = G.hpr[lane - 75];
  else if (lane < 125) sG[lane] = G.hpwr[lane - 100];
}
// the hprime / hprimewgll table an element uses (folded ones on regular elements in FMA builds)
__device__ __forceinline__ const realw* gll_hp(const realw* sG, bool irr) { return (SF_FOLD && !irr) ? sG + 75 : sG; }
__device__ __forceinline__ const realw* gll_hpw(const realw* sG, bool irr) {
  return (SF_FOLD && !irr) ? sG + 100 : sG + 25;
}

// One line of five GLL points against the derivative tables, held by one lane: the coefficients have
// constant indices and come from scalar registers, and each point of the line is read once instead
// of once per output. Sums left to right, as tile_gradient and tile_divergence.
__device__ __forceinline__ void line_gradient(const GLLk& G, const realw in[5], realw out[5]) {
#pragma unroll
  for (int m = 0; m < 5; m++) {
    realw r = sum2(G.hp[m * 5], in[0], G.hp[m * 5 + 1], in[1]);
#pragma unroll
    for (int l = 2; l < 5; l++) r = add_product(r, G.hp[m * 5 + l], in[l]);
    out[m] = r;
  }
}
__device__ __forceinline__ void line_divergence(const GLLk& G, const realw in[5], realw out[5]) {
#pragma unroll
  for (int m = 0; m < 5; m++) {
    realw r = sum2(G.hpw[m], in[0], G.hpw[5 + m], in[1]);
#pragma unroll
    for (int l = 2; l < 5; l++) r = add_product(r, G.hpw[l * 5 + m], in[l]);
    out[m] = r;
  }
}

__device__ __forceinline__ JacPt load_jac(const realw* J, int64_t P, int64_t q) {
  JacPt r;
  r.xix = J[q]; r.xiy = J[P + q]; r.xiz = J[2 * P + q];
  r.etax = J[3 * P + q]; r.etay = J[4 * P + q]; r.etaz = J[5 * P + q];
  r.gax = J[6 * P + q]; r.gay = J[7 * P + q]; r.gaz = J[8 * P + q];
  r.jac = J[9 * P + q];
  return r;
}

}  // namespace sf
