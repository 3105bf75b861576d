// Ray-cast renderer: drawSimBVHKernelManyEnvs + meshQueryRayManyEnvs +
// downsample_kernel (render.py:276-498, 699-724) and the vertex normals
// (render.py:81-121).
//
// Three traversals give the same images bit for bit.  The automatic one is the
// block form below: a wavefront walks the BVH once for a block of rays.  The
// other two trace rays one by one, with a stack in LDS (slot-major, so the 64
// lanes of a slot fall in distinct banks): one ray per lane, or a lane per
// pixel with its quad of 2x-supersampled rays.  The 2x2 box filter sums a
// pixel's rays in the reference's order, so no ray buffer goes to HBM.
// Traversal order, the Moller-Trumbore test and the strict "0 < t < tMin"
// acceptance follow the reference expression by expression for every ray, and
// the box tests' decisions equal the reference's slab test (a fast form with
// an exact fallback, render_box.hpp), so hit triangles are bit-exact.
#include <algorithm>
#include <climits>
#include <type_traits>

#include "common.hpp"
#include "render_box.hpp"

namespace ffsrl {

constexpr int kStack = 32;  // deepest supported BVH (levels); the reference's stack size
constexpr int kWaves = 1;   // wavefronts per block (one 8x8 ray tile each)
constexpr int kXcds = 8;    // gfx950 dispatches workgroups round-robin over 8 XCDs

__device__ __forceinline__ float mt_isect(f3 a, f3 b, f3 c, f3 o, f3 d) {
  const f3 e1 = b - a, e2 = c - a;
  const f3 pv = cross(d, e2);
  const float det = dot(e1, pv);
  if (fabsf(det) < 0.0001f) return -1.0f;
  const float inv = 1.0f / det;
  const f3 tv = o - a;
  const float u = dot(tv, pv) * inv;
  if (u < 0.0f || u > 1.0f) return -1.0f;
  const f3 qv = cross(tv, e1);
  const float v = dot(d, qv) * inv;
  if (v < 0.0f || u + v > 1.0f) return -1.0f;
  return dot(e2, qv) * inv;
}

template <typename T>
__device__ __forceinline__ T ldu4(const T* base, int i) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + (uint32_t)i * (uint32_t)sizeof(T));
}

// float -> int as the reference's int() on the device: truncation toward
// zero, NaN to 0, saturating at the int range.
__device__ __forceinline__ int trunc_i(float x) {
  if (!(x == x)) return 0;
  if (x >= 2147483647.0f) return 2147483647;
  if (x <= -2147483648.0f) return -2147483647 - 1;
  return (int)x;
}

// One texel of the concatenated table; an index outside it reads as zero
// (the reference's lookup reads one column past a texture's last, where the
// weight is zero).
__device__ __forceinline__ f3 texel(const ffsrl_batch& b, int64_t i) {
  if (i < 0 || i >= b.n_texels) return mk(0.0f, 0.0f, 0.0f);
  return xyz(ld4(b.texels, i));
}

// texture_interpolation (render.py:124-148): bilinear lookup in square
// texture tx at texture coordinates (s, t), with the reference's indexing
// y + x * width and no clamp of x0 + 1 / y0 + 1.
__device__ __forceinline__ f3 texture_lookup(const ffsrl_batch& b, int tx, float s, float t) {
  const int64_t first = b.tex_info[2 * tx];
  const int size = (int)b.tex_info[2 * tx + 1];
  const float fx = s * (float)(size - 1), fy = (1.0f - t) * (float)(size - 1);
  const int x0 = trunc_i(fx), y0 = trunc_i(fy);
  const int x1 = x0 + 1, y1 = y0 + 1;
  const float ax = fx - (float)x0, ay = fy - (float)y0;
  const f3 c00 = texel(b, first + y0 + (int64_t)x0 * size), c10 = texel(b, first + y0 + (int64_t)x1 * size);
  const f3 c01 = texel(b, first + y1 + (int64_t)x0 * size), c11 = texel(b, first + y1 + (int64_t)x1 * size);
  const f3 lower = c00 * (1.0f - ax) + c10 * ax;
  const f3 upper = c01 * (1.0f - ax) + c11 * ax;
  return lower * (1.0f - ay) + upper * ay;
}

// One ray's traversal: right-first depth-first over the env's BVH, strict
// 0 < t < tMin, as meshQueryRayManyEnvs (render.py:430-496).  stk is the
// lane's column of a slot-major stack in LDS.
struct RayHit {
  float t;   // 1e6: no hit
  int best;  // leaf-order triangle
};

__device__ __forceinline__ RayHit trace_ray(const float4* blo, const float4* bhi, const int4* tris, const float4* X,
                                            f3 o, f3 d, f3 inv, bool ray_ok, int* stk, int depth) {
  stk[0] = 0;
  int count = 1, best = -1;
  float tMin = 1e6f;
  while (count) {
    const int node = stk[(count - 1) * 64];
    count -= 1;
    const float4 lo = ldu4(blo, node), hi = ldu4(bhi, node);
    if (visit_node(o, d, inv, xyz(lo), xyz(hi), tMin, ray_ok)) {
      const int n = __float_as_int(hi.w);
      if (n > 0) {
        const int first = __float_as_int(lo.w);
        for (int k = 0; k < n; ++k) {
          const int4 t = ldu4(tris, first + k);
          const float tt = mt_isect(xyz(ldu4(X, t.x)), xyz(ldu4(X, t.y)), xyz(ldu4(X, t.z)), o, d);
          if (tt < tMin && tt > 0.0f) {
            tMin = tt;
            best = first + k;
          }
        }
      } else if (count + 2 <= depth) {  // depth = deepest BVH level + 1: never false
        const int l = __float_as_int(lo.w);
        stk[count * 64] = l;
        stk[(count + 1) * 64] = l + 1;
        count += 2;
      }
    }
  }
  return RayHit{tMin, best};
}

struct RenderOut {
  float* depth;
  float* rgb;
  const float* normals;
  const float* vcolor;
  const float* tcolor;
  int32_t* hit;
  float* thit;
};

// Shading of one ray's hit (colour modes; mode 4 gives depth in .x):
// render.py:356-409, expression by expression.
__device__ __forceinline__ f3 shade(const ffsrl_batch& b, const ffsrl_camera& cam, const RenderOut& out, int64_t vb,
                                    int64_t fb, f3 o, f3 d, float tMin, int best, int4 tri) {
  f3 color;
  if (cam.mode == 4) {
    const float c = tMin / 50.0f * 1.0f;
    color = mk(c, c, c);
  } else {
    const f3 A = xyz(ld4(b.x, vb + tri.x)), B = xyz(ld4(b.x, vb + tri.y)), C = xyz(ld4(b.x, vb + tri.z));
    const f3 p = o + d * tMin;
    const float area = length(cross(B - A, C - A));
    const float w = length(cross(B - A, p - A)) / area;
    const float v = length(cross(p - A, C - A)) / area;
    const float u = 1.0f - w - v;
    const f3 na = xyz(ld4(out.normals, vb + tri.x)), nb = xyz(ld4(out.normals, vb + tri.y)),
             nc = xyz(ld4(out.normals, vb + tri.z));
    const f3 normal = (na * u + nb * v) + nc * w;
    if (cam.mode == 2) {
      color = normal * 0.5f + mk(0.5f, 0.5f, 0.5f);
    } else {
      const int tex = (cam.mode == 1 && b.tri_tex) ? b.tri_tex[fb + best] : -1;
      if (cam.mode == 0) {
        color = mk(1.0f, 1.0f, 1.0f);
      } else if (cam.mode == 5) {
        const float* tc = out.tcolor + 3 * (int64_t)(fb + best);
        color = mk(tc[0], tc[1], tc[2]);
      } else if (tex >= 0) {  // texture mode: tex = u * tex_a + v * tex_b + w * tex_c (render.py:356-377)
        const float* uv = b.tri_uv + 6 * (int64_t)(fb + best);
        const float s = (u * uv[0] + v * uv[2]) + w * uv[4];
        const float t = (u * uv[1] + v * uv[3]) + w * uv[5];
        color = texture_lookup(b, tex, s, t);
      } else {  // vertex colour, and the texture mode's fallback (render.py:378-380)
        const float* ca = out.vcolor + 3 * (vb + tri.x);
        const float* cb = out.vcolor + 3 * (vb + tri.y);
        const float* cc = out.vcolor + 3 * (vb + tri.z);
        color = ((mk(ca[0], ca[1], ca[2]) + mk(cb[0], cb[1], cb[2])) + mk(cc[0], cc[1], cc[2])) / 3.0f;
      }
      float val = cam.light_intensity * dot(normal, mk(cam.light_dir[0], cam.light_dir[1], cam.light_dir[2]));
      if (val < 0.0f) val = 0.0f;
      const float lambert = 0.0f + val;
      color = color * lambert;
    }
  }
  if (color.x > 1.0f) color.x = 1.0f;
  if (color.y > 1.0f) color.y = 1.0f;
  if (color.z > 1.0f) color.z = 1.0f;
  return color;
}

// Outputs of one ray (a lane of an 8x8-ray tile): hit and distance, shading,
// and the 2x2 box filter across lanes.
__device__ __forceinline__ void finish_ray(const ffsrl_batch& b, const ffsrl_camera& cam, const RenderOut& out,
                                           int lane, int64_t oi, int64_t rays_env, int r, int row, int col,
                                           int64_t vb, int64_t fb, f3 o, f3 d, float tMin, int best) {
  const bool hitp = tMin < 1e6f;
  int4 tri = make_int4(0, 0, 0, -1);
  if (hitp) tri = ldi4(b.tris, fb + best);
  if (out.hit) out.hit[oi * rays_env + r] = hitp ? tri.w : -1;
  if (out.thit) out.thit[oi * rays_env + r] = hitp ? tMin : 0.0f;

  const f3 color = hitp ? shade(b, cam, out, vb, fb, o, d, tMin, best, tri) : mk(0.0f, 0.0f, 0.0f);
  // 2x2 box: rays (2py+i, 2px+j) summed in (i, j) = (0,0), (0,1), (1,0), (1,1) order.
  const bool owner = ((lane & 1) == 0) && (((lane >> 3) & 1) == 0);
  const int64_t pix = oi * cam.height * cam.width + (row >> 1) * cam.width + (col >> 1);
  if (cam.mode == 4) {
    const float c01 = __shfl_down(color.x, 1), c10 = __shfl_down(color.x, 8), c11 = __shfl_down(color.x, 9);
    if (owner && out.depth) out.depth[pix] = (((color.x + c01) + c10) + c11) / 4.0f;
  } else {
    float ch[3] = {color.x, color.y, color.z};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const float c01 = __shfl_down(ch[k], 1), c10 = __shfl_down(ch[k], 8), c11 = __shfl_down(ch[k], 9);
      if (owner && out.rgb) out.rgb[3 * pix + k] = (((ch[k] + c01) + c10) + c11) / 4.0f;
    }
    if (out.depth) {
      // RGB-D: the depth image of the same hits, computed as depth mode does
      float dz = 0.0f;
      if (hitp) {
        dz = tMin / 50.0f * 1.0f;
        if (dz > 1.0f) dz = 1.0f;
      }
      const float d01 = __shfl_down(dz, 1), d10 = __shfl_down(dz, 8), d11 = __shfl_down(dz, 9);
      if (owner) out.depth[pix] = (((dz + d01) + d10) + d11) / 4.0f;
    }
  }
}

// A stack entry is a node id (< 2^28) and, in its top 4 bits, the rays of
// the lane's quad whose own traversal reaches the node (they hit its parent).
constexpr int kQuadShift = 28;
constexpr int kNodeMask = (1 << kQuadShift) - 1;
// Images from this size refuse BVHs that a quad entry cannot hold, unless one
// ray per lane is asked for.
constexpr int kQuadMinPixels = 128 * 128;

// Environments: env_begin + el for el < n_env, or list[el] when list is not
// NULL; outputs are indexed by el for a range and by the env id for a list.
//
// One lane renders one pixel: its quad of supersampled rays k = 0..3, ray
// (2 py + (k >> 1), 2 px + (k & 1)).  The quad shares one traversal stack
// whose entries carry the mask of quad rays that reach the node: a node is
// tested for exactly those rays, and its children are pushed with the rays
// that hit it.  Every ray therefore tests the nodes of its own right-first
// DFS, in the same order and against its own tMin, so its hits are those of
// a traversal of its own; the quad shares the node and triangle loads, the
// stack and the loop.  A wavefront takes an 8x8-pixel tile of one env.
__global__ __launch_bounds__(64 * kWaves) void k_render_quad(ffsrl_batch b, ffsrl_camera cam, int env_begin,
                                                             const int32_t* list, int n_env, RenderOut out,
                                                             int depth) {
  extern __shared__ int stack[];  // [kWaves][depth][64]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int RW = 2 * cam.width;
  const int tiles_x = (cam.width + 7) >> 3, tiles = tiles_x * ((cam.height + 7) >> 3);
  // XCD-aware mapping of the 1D grid: block B runs on XCD B % 8, so the
  // blocks of env el are B = 8 * (bpe * (el / 8) + j) + el % 8, j < bpe: all
  // tiles of an env share one XCD's L2 (its BVH, triangles and positions are
  // fetched into one L2 instead of eight).
  const int bpe = (tiles + kWaves - 1) / kWaves;
  const int xcd = blockIdx.x % kXcds, k = blockIdx.x / kXcds;
  const int el = (k / bpe) * kXcds + xcd;
  const int tile = (k % bpe) * kWaves + wave;
  if (el >= n_env || tile >= tiles) return;  // whole wavefront exits; no block barrier below
  const int px = (tile % tiles_x) * 8 + (lane & 7), py = (tile / tiles_x) * 8 + (lane >> 3);
  if (px >= cam.width || py >= cam.height) return;  // no cross-lane operation below
  const int env = list ? list[el] : env_begin + el;
  const int64_t oi = list ? env : el;  // output slot
  const ffsrl_env_desc e = b.envs[env];
  const int64_t vb = e.vbase, sb = e.boundbase, fb = e.fbase;
  const f3 o = mk(cam.origin[0], cam.origin[1], cam.origin[2]);
  f3 d[4], inv[4];
  bool ray_ok[4];
  float tMin[4];
  int best[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = (2 * py + (q >> 1)) * RW + 2 * px + (q & 1);
    d[q] = xyz(ld4(cam.dirs, r));
    inv[q] = mk(1.0f / d[q].x, 1.0f / d[q].y, 1.0f / d[q].z);
    ray_ok[q] = ray_dir_ok(d[q]);
    tMin[q] = 1e6f;
    best[q] = -1;
  }

  // env-uniform bases; node / triangle / vertex ids are non-negative int32,
  // so loads take a 32-bit unsigned offset from a scalar base
  const float4* blo = reinterpret_cast<const float4*>(b.bvh_lo) + sb;
  const float4* bhi = reinterpret_cast<const float4*>(b.bvh_hi) + sb;
  const int4* tris = reinterpret_cast<const int4*>(b.tris) + fb;
  const float4* X = reinterpret_cast<const float4*>(b.x) + vb;
  int* stk = stack + wave * depth * 64 + lane;
  stk[0] = 0xF << kQuadShift;  // the root, reached by all four rays
  int count = 1;
  while (count) {
    const int entry = stk[(count - 1) * 64];
    count -= 1;
    const int node = entry & kNodeMask, reach = (int)((unsigned)entry >> kQuadShift);
    const float4 lo = ldu4(blo, node), hi = ldu4(bhi, node);
    int hits = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (((reach >> q) & 1) && visit_node(o, d[q], inv[q], xyz(lo), xyz(hi), tMin[q], ray_ok[q])) hits |= 1 << q;
    if (!hits) continue;
    const int n = __float_as_int(hi.w);
    if (n > 0) {
      const int first = __float_as_int(lo.w);
      for (int k2 = 0; k2 < n; ++k2) {
        const int4 t = ldu4(tris, first + k2);
        const f3 A = xyz(ldu4(X, t.x)), B = xyz(ldu4(X, t.y)), C = xyz(ldu4(X, t.z));
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if (!((hits >> q) & 1)) continue;
          const float tt = mt_isect(A, B, C, o, d[q]);
          if (tt < tMin[q] && tt > 0.0f) {
            tMin[q] = tt;
            best[q] = first + k2;
          }
        }
      }
    } else if (count + 2 <= depth) {  // depth = deepest BVH level + 1: never false
      const int l = __float_as_int(lo.w);
      stk[count * 64] = l | (hits << kQuadShift);
      stk[(count + 1) * 64] = (l + 1) | (hits << kQuadShift);
      count += 2;
    }
  }

  const int64_t rays_env = (int64_t)RW * 2 * cam.height;
  const int64_t pix = oi * cam.height * cam.width + (int64_t)py * cam.width + px;
  f3 color[4];
  float dz[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const bool hitp = tMin[q] < 1e6f;
    int4 tri = make_int4(0, 0, 0, -1);
    if (hitp) tri = ldi4(b.tris, fb + best[q]);
    const int64_t r = (int64_t)(2 * py + (q >> 1)) * RW + 2 * px + (q & 1);
    if (out.hit) out.hit[oi * rays_env + r] = hitp ? tri.w : -1;
    if (out.thit) out.thit[oi * rays_env + r] = hitp ? tMin[q] : 0.0f;
    color[q] = hitp ? shade(b, cam, out, vb, fb, o, d[q], tMin[q], best[q], tri) : mk(0.0f, 0.0f, 0.0f);
    dz[q] = 0.0f;
    if (hitp) {
      dz[q] = tMin[q] / 50.0f * 1.0f;
      if (dz[q] > 1.0f) dz[q] = 1.0f;
    }
  }
  // 2x2 box: rays (2py+i, 2px+j) summed in (i, j) = (0,0), (0,1), (1,0), (1,1) order.
  if (cam.mode == 4) {
    if (out.depth) out.depth[pix] = (((color[0].x + color[1].x) + color[2].x) + color[3].x) / 4.0f;
  } else {
    if (out.rgb) {
      out.rgb[3 * pix + 0] = (((color[0].x + color[1].x) + color[2].x) + color[3].x) / 4.0f;
      out.rgb[3 * pix + 1] = (((color[0].y + color[1].y) + color[2].y) + color[3].y) / 4.0f;
      out.rgb[3 * pix + 2] = (((color[0].z + color[1].z) + color[2].z) + color[3].z) / 4.0f;
    }
    // RGB-D: the depth image of the same hits, computed as depth mode does
    if (out.depth) out.depth[pix] = (((dz[0] + dz[1]) + dz[2]) + dz[3]) / 4.0f;
  }
}

// Environments: env_begin + el for el < n_env, or list[el] when list is not
// NULL; outputs are indexed by el for a range and by the env id for a list.
//
// Per-ray form: one lane per supersampled ray, a wavefront per 8x8-ray tile;
// the 2x2 box filter sums across lanes with shuffles.
__global__ __launch_bounds__(64 * kWaves) void k_render(ffsrl_batch b, ffsrl_camera cam, int env_begin,
                                                        const int32_t* list, int n_env, RenderOut out, int depth) {
  extern __shared__ int stack[];  // [kWaves][depth][64]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int RW = 2 * cam.width, RH = 2 * cam.height;
  const int tiles_x = RW >> 3, tiles = tiles_x * (RH >> 3);
  // XCD-aware mapping of the 1D grid: block B runs on XCD B % 8, so the
  // blocks of env el are B = 8 * (bpe * (el / 8) + j) + el % 8, j < bpe: all
  // tiles of an env share one XCD's L2 (its BVH, triangles and positions are
  // fetched into one L2 instead of eight).
  const int bpe = (tiles + kWaves - 1) / kWaves;
  const int xcd = blockIdx.x % kXcds, k = blockIdx.x / kXcds;
  const int el = (k / bpe) * kXcds + xcd;
  const int tile = (k % bpe) * kWaves + wave;
  if (el >= n_env || tile >= tiles) return;  // whole wavefront exits; no block barrier below
  const int env = list ? list[el] : env_begin + el;
  const int64_t oi = list ? env : el;  // output slot
  const int col = (tile % tiles_x) * 8 + (lane & 7), row = (tile / tiles_x) * 8 + (lane >> 3);
  const int r = row * RW + col;
  const ffsrl_env_desc e = b.envs[env];
  const int64_t vb = e.vbase, sb = e.boundbase, fb = e.fbase;
  const f3 o = mk(cam.origin[0], cam.origin[1], cam.origin[2]);
  const f3 d = xyz(ld4(cam.dirs, r));
  const f3 inv = mk(1.0f / d.x, 1.0f / d.y, 1.0f / d.z);
  const bool ray_ok = ray_dir_ok(d);

  // env-uniform bases; node / triangle / vertex ids are non-negative int32,
  // so loads take a 32-bit unsigned offset from a scalar base
  const float4* blo = reinterpret_cast<const float4*>(b.bvh_lo) + sb;
  const float4* bhi = reinterpret_cast<const float4*>(b.bvh_hi) + sb;
  const int4* tris = reinterpret_cast<const int4*>(b.tris) + fb;
  const float4* X = reinterpret_cast<const float4*>(b.x) + vb;
  int* stk = stack + wave * depth * 64 + lane;
  const RayHit h = trace_ray(blo, bhi, tris, X, o, d, inv, ray_ok, stk, depth);
  const float tMin = h.t;
  const int best = h.best;
  finish_ray(b, cam, out, lane, oi, (int64_t)RW * RH, r, row, col, vb, fb, o, d, tMin, best);
}

// ---------------------------------------------------------------------------
// Block form: one wavefront renders a block of SW x SH subtiles of 8x8 rays of
// one env (a lane holds one ray of each subtile).  All rays share the origin,
// so the rays of a block lie in a narrow cone, and the wavefront walks the BVH
// once for the cone, a node per lane, instead of once per ray: it collects the
// triangles of the leaf boxes that the cone meets, finds for each (a triangle
// per lane) the subtiles that it can cover, and tests those subtiles' rays, a
// ray per lane, against the triangle's data broadcast from LDS.
//
// The hits are those of the per-ray traversal (trace_ray), bit for bit:
// - Bounds are min / max of their children's, and the slab values are
//   monotone in the bounds, so a ray that passes a leaf's box test passes its
//   ancestors'.  The per-ray traversal therefore tests exactly the triangles
//   of the leaves whose box test the ray passes with the tMin it has by then.
// - Let t be the least distance that the intersection test (mt_isect)
//   returns, and every other triangle's distance be beyond t and beyond the
//   entry tb of that leaf's box.  tMin is t or more until the leaf is reached
//   and beyond tb, so the leaf is visited and its triangle is the hit.  A ray
//   for which this cannot be shown (ties, grazing boxes, zero or tiny direction
//   components) is traced by trace_ray.
// - Culling and the first test of a triangle are conservative.  The terms of
//   mt_isect are linear in the direction: det = d . (e2 x e1), u det =
//   d . (e2 x tv), v det = d . (tv x e1).  Their signs decide a ray's miss or
//   hit where they exceed the rounding of both evaluations; a ray within it
//   takes mt_isect itself.  The nearest triangle's t comes from mt_isect.
// - The directions are checked to lie on a grid p0 + col B + row C (the
//   camera's pinhole table does); rays of any other table, and rays that meet
//   bounds which are not finite, are traced by trace_ray.
//
// Bound: VALU issue (a 2x2 block of 64x64 depth images of mixed 1k-40k-tet
// scenes: 4.5k instructions, half of them tests of 46 triangles against 1.2 of
// its 4 subtiles each, the rest the walk of 5 steps, 1.1 batches and the exact
// checks; per ray the traversal kernels took 2.3k for a quarter of that block,
// for about 40 dependent node visits).  Two levels of the tree per step halve
// the walk's dependent loads; a triangle's terms are set up once for a block
// and read from LDS by broadcast; 5 wavefronts per SIMD (96 VGPRs) hide both
// (4 were 10% slower, 6 spill).  Measured, per-ray / quad traversal against
// this: 64x64 depth of 768 mixed scenes 693 -> 419 us, of 1024 liver scenes
// 1451 -> 428; 128x128 RGB-D of 384 20k-tet ellipsoids 1272 -> 653; 128x128
// depth of one cube 125 -> 26.
constexpr int kTileStack = 384;  // inner nodes' children waiting in the walk
constexpr int kTileList = 256;   // triangles found and not yet tested
constexpr int kTileGridBytes = 128;
constexpr int kTileListBytes = kTileList * 8;
constexpr int kTileWorkBytes = 64 * 64 + kTileStack * 4;  // a batch's triangles, the walk's stack; or trace_ray's stacks

__device__ __forceinline__ float fdot(f3 a, f3 b) { return fmaf(a.x, b.x, fmaf(a.y, b.y, a.z * b.z)); }
__device__ __forceinline__ f3 fcross(f3 a, f3 b) {
  return mk(fmaf(a.y, b.z, -(a.z * b.y)), fmaf(a.z, b.x, -(a.x * b.z)), fmaf(a.x, b.y, -(a.y * b.x)));
}
__device__ __forceinline__ f3 fmad(f3 a, float s, f3 b) {
  return mk(fmaf(a.x, s, b.x), fmaf(a.y, s, b.y), fmaf(a.z, s, b.z));
}
__device__ __forceinline__ f3 funit(f3 a) { return a * __builtin_amdgcn_rsqf(fdot(a, a)); }
__device__ __forceinline__ float l1(f3 a) { return fabsf(a.x) + fabsf(a.y) + fabsf(a.z); }
__device__ __forceinline__ float ufirst(float v) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}
__device__ __forceinline__ f3 ufirst(f3 a) { return mk(ufirst(a.x), ufirst(a.y), ufirst(a.z)); }
__device__ __forceinline__ int lanes_below(unsigned long long m) {
  return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// The axis f of a pinhole table, from its corner rays: the points a00 d00,
// a10 d10, a01 d01, a11 d11 of the image plane form a parallelogram, which
// gives the a's up to a common factor, and f is the plane's normal.
__device__ __forceinline__ f3 image_axis(f3 d00, f3 d10, f3 d01, f3 d11) {
  const f3 k = fcross(d01, d11);
  const float r = 1.0f / fdot(d10, k);
  const f3 x = d10 * (fdot(d00, k) * r) - d00;                    // a10 d10 - d00, with a00 = 1
  const f3 y = d01 * (fdot(d10, fcross(d00, d11)) * r) - d00;     // a01 d01 - d00
  const f3 n = funit(fcross(x, y));
  return ufirst(fdot(n, d00) < 0.0f ? -n : n);
}

// The block's rays: the direction at (col, row) is that of p0 + col B + row C,
// a point of a plane normal to the axis f, at distance about 1.
struct RayGrid {
  f3 p0, B, C;
  f3 f;    // the axis over its product with c: dot(f, p) = 1 (not kept in LDS)
  f3 c;    // unit, within the block
  f3 n[4]; // side planes: dot(n, p) <= 0 inside
};
constexpr float kGridSlack = 1.5e-6f;  // a ray may miss its grid point by this, per component
constexpr float kConeTilt = 1e-5f;     // boxes are tested against planes tilted outward by this

// From the directions of the block's corners (00, last column, last row, both).
__device__ __forceinline__ RayGrid make_grid(f3 axis, f3 d00, f3 d10, f3 d01, f3 d11, int cols, int rows) {
  RayGrid g;
  g.c = ufirst(funit((d00 + d10) + (d01 + d11)));
  g.f = ufirst(axis * (1.0f / fdot(axis, g.c)));
  const f3 p0 = d00 * (1.0f / fdot(d00, g.f)), p1 = d10 * (1.0f / fdot(d10, g.f)), p2 = d01 * (1.0f / fdot(d01, g.f));
  g.p0 = ufirst(p0);
  g.B = ufirst((p1 - p0) * (1.0f / (float)(cols - 1)));
  g.C = ufirst((p2 - p0) * (1.0f / (float)(rows - 1)));
  f3 n[4] = {fcross(g.p0, g.C), fcross(p1, g.C), fcross(g.p0, g.B), fcross(p2, g.B)};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    n[i] = funit(n[i]);
    if (fdot(n[i], g.c) > 0.0f) n[i] = -n[i];
    g.n[i] = ufirst(n[i]);
  }
  return g;
}

// A unit direction on its grid point, which is at distance 1 to within 7%.
__device__ __forceinline__ bool on_grid(const RayGrid& g, f3 d, int col, int row) {
  const float k = fdot(d, g.f);
  const f3 p = d * __builtin_amdgcn_rcpf(k), q = fmad(g.C, (float)row, fmad(g.B, (float)col, g.p0));
  const float off = fmaxf(fmaxf(fabsf(p.x - q.x), fabsf(p.y - q.y)), fabsf(p.z - q.z));
  return off <= kGridSlack && k > 0.93f && k < 1.07f && fdot(d, g.c) > 0.9f && fabsf(fdot(d, d) - 1.0f) <= 4e-6f;
}

__device__ __forceinline__ void put_grid(float4* w, const RayGrid& g) {
  w[0] = make_float4(g.p0.x, g.p0.y, g.p0.z, g.c.x);
  w[1] = make_float4(g.B.x, g.B.y, g.B.z, g.c.y);
  w[2] = make_float4(g.C.x, g.C.y, g.C.z, g.c.z);
#pragma unroll
  for (int i = 0; i < 4; ++i) w[3 + i] = make_float4(g.n[i].x, g.n[i].y, g.n[i].z, 0.0f);
}
__device__ __forceinline__ RayGrid get_grid(const float4* w) {
  RayGrid g;
  const float4 a = w[0], b = w[1], c = w[2];
  g.p0 = xyz(a);
  g.B = xyz(b);
  g.C = xyz(c);
  g.c = mk(a.w, b.w, c.w);
#pragma unroll
  for (int i = 0; i < 4; ++i) g.n[i] = xyz(w[3 + i]);
  return g;
}

// 1: the box lies outside the block's cone; 0: it may meet it; -1: bounds that
// are not finite.  A ray's box test rounds by a few 1e-7 of the distance,
// against kConeTilt; the slack covers the rounding of this evaluation relative
// to the box's corners.  (Box centre and extent are taken twice as large.)
__device__ __forceinline__ int box_outside(const RayGrid& g, f3 o, float4 lo, float4 hi) {
  const f3 l = xyz(lo) - o, h = xyz(hi) - o;
  const f3 c = l + h, e = h - l;
  const float size = l1(c) + l1(e);
  const float slack = 2e-6f * size;
  auto extent = [&](f3 n, float s) {  // s |n| . |e|
    return s * fmaf(fabsf(n.x), fabsf(e.x), fmaf(fabsf(n.y), fabsf(e.y), fabsf(n.z) * fabsf(e.z)));
  };
  const float far = fdot(g.c, c) + extent(g.c, 1.0f);  // extent along the centre direction
  bool out = far < -slack;                             // behind the origin
  const float edge = fmaf(kConeTilt, fabsf(far), slack);
#pragma unroll
  for (int i = 0; i < 4; ++i) out = out | (fdot(g.n[i], c) - extent(g.n[i], 1.0f) > edge);
  return size < 3e38f ? (int)out : -1;
}

struct TileLds {
  float4* grid; // the block's RayGrid: kept here, not in registers, between uses
  int2* list;   // (leaf-order triangle, leaf node)
  float4* tri;  // 4 per triangle of a batch
  int* stack;   // left children of inner nodes that the cone meets
};

// A box test's outcome for the wavefront: met inner nodes go to the stack, met
// leaves' triangles to the list.  False when the list would overflow.
__device__ __forceinline__ bool take_nodes(const TileLds& L, int node, float4 lo, float4 hi, bool met, int& ns,
                                           int& nl) {
  const int n = __float_as_int(hi.w), first = __float_as_int(lo.w);
  const unsigned long long inner = __ballot(met && n <= 0);
  if (met && n <= 0) L.stack[ns + lanes_below(inner)] = first;
  ns += __popcll(inner);
  for (int j = 0;; ++j) {
    const unsigned long long leaf = __ballot(met && j < n);
    if (!leaf) return true;
    if (nl + __popcll(leaf) > kTileList) return false;
    if (met && j < n) L.list[nl + lanes_below(leaf)] = make_int2(first + j, node);
    nl += __popcll(leaf);
  }
}

// One step of the walk, two levels at a time: of at most 16 inner nodes from
// the top of the stack, the four grandchildren are tested by four lanes (a
// child that is a leaf by the first of its two).  False when the stack or the
// list would overflow, or bounds are not finite.
__device__ __forceinline__ bool walk_step(f3 o, const float4* blo, const float4* bhi,
                                          const TileLds& L, int& ns, int& nl) {
  const int lane = threadIdx.x & 63;
  const int take = ns < 16 ? ns : 16;
  if (ns - take + 64 > kTileStack) return false;
  bool on = (lane >> 2) < take;
  int node = on ? L.stack[ns - take + (lane >> 2)] + ((lane >> 1) & 1) : 0;
  ns -= take;
  float4 lo = ldu4(blo, node), hi = ldu4(bhi, node);
  if (__any(on && !(l1(xyz(lo)) + l1(xyz(hi)) < 3e38f))) return false;
  if (__float_as_int(hi.w) <= 0) {
    node = on ? __float_as_int(lo.w) + (lane & 1) : 0;
    lo = ldu4(blo, node);
    hi = ldu4(bhi, node);
  } else {
    on = on && (lane & 1) == 0;
  }
  const int outside = box_outside(get_grid(L.grid), o, lo, hi);
  if (__any(on && outside < 0)) return false;
  __syncthreads();  // the stack entries are read before others overwrite them
  const bool fits = take_nodes(L, node, lo, hi, on && outside == 0, ns, nl);
  __syncthreads();
  return fits;
}

// The ray of one subtile.  [lo, hi] bounds what mt_isect returns for the
// triangle of least lower bound so far (its leaf-order id and leaf); lo2 is the
// least lower bound of the others.
struct TileRay {
  f3 d;
  float lo, hi, lo2;
  int best, leaf;
};

// One triangle of a batch, as the lanes read it.
struct TileTri {
  f3 nd, nu, nv;    // det, u det and v det by direction
  float key;        // no ray of the block has a distance below
  float m;          // rounding of the three terms and of those of mt_isect
  float tn, rel;    // t = tn / det; relative rounding of t
  int id, leaf;
  float det0;       // mt_isect's least |det|, plus rounding
};

__device__ __forceinline__ TileTri read_tri(const float4* w) {
  const float4 a = w[0], b = w[1], c = w[2], e = w[3];
  return TileTri{xyz(a), xyz(b), xyz(c), a.w, b.w, c.w, e.x, __float_as_int(e.y), __float_as_int(e.z), e.w};
}

// Tests one triangle against the rays of one subtile.
__device__ __forceinline__ void test_tri(const TileTri& w, TileRay& ray, f3 o, const int4* tris, const float4* X) {
  if (!__any(!(w.key > ray.hi))) return;  // beyond every ray's nearest
  const float det = fdot(w.nd, ray.d), un = fdot(w.nu, ray.d), vn = fdot(w.nv, ray.d);
  const float sg = copysignf(1.0f, det);
  const float us = un * sg, vs = vn * sg, ws = (fabsf(det) - us) - vs;
  const float in = fminf(fminf(us, vs), ws);  // > 0 inside the triangle
  const bool out = in < -w.m;
  if (__all(out)) return;
  const bool sure = (in > w.m) & (fabsf(det) > w.det0);
  float t = w.tn * __builtin_amdgcn_rcpf(det);
  float lo = fmaf(-t, w.rel, t), hi = fmaf(t, w.rel, t);
  bool hit = sure & (t > 0.0f);
  const bool maybe = !out & !sure;  // within rounding of an edge or of the least det
  if (__any(maybe)) {
    if (maybe) {
      const int4 q = ldu4(tris, w.id);
      t = mt_isect(xyz(ldu4(X, q.x)), xyz(ldu4(X, q.y)), xyz(ldu4(X, q.z)), o, ray.d);
      lo = hi = t;
      hit = t > 0.0f;
    }
  }
  lo = hit ? lo : 3e38f;
  const bool near = lo < ray.lo;
  ray.lo2 = __builtin_amdgcn_fmed3f(lo, ray.lo, ray.lo2);  // ray.lo <= ray.lo2
  ray.lo = near ? lo : ray.lo;
  ray.hi = near ? hi : ray.hi;
  ray.best = near ? w.id : ray.best;
  ray.leaf = near ? w.leaf : ray.leaf;
}

// Tests list entries l0 .. l0 + n - 1 (n <= 64) against the block's rays:
// first a triangle per lane against the subtiles' corners, then the
// remaining ones, front faces first (they hide the back faces of a closed
// surface), against the subtiles that they can cover.
template <int SW, int SH>
__device__ __forceinline__ void test_batch(f3 o, const int4* tris, const float4* X, const TileLds& L, int l0, int n,
                                           TileRay (&ray)[SW * SH]) {
  const RayGrid g = get_grid(L.grid);
  const int lane = threadIdx.x & 63;
  const bool on = lane < n;
  const int2 ent = L.list[on ? l0 + lane : l0];
  const int4 t = ldu4(tris, ent.x);
  const f3 a = xyz(ldu4(X, t.x)), b = xyz(ldu4(X, t.y)), c = xyz(ldu4(X, t.z));
  const f3 e1 = b - a, e2 = c - a, tv = o - a;  // as mt_isect rounds them
  const f3 nd = fcross(e2, e1), nu = fcross(e2, tv), nv = fcross(tv, e1);
  const float tn = dot(e2, cross(tv, e1));      // mt_isect's
  const float s1 = l1(e1), s2 = l1(e2), st = l1(tv);
  const float s12 = s1 * s2, su = st * s2, sv = st * s1;
  // det over the block: its sign, where it does not change
  constexpr float kM = 2e-5f;  // rays off their grid points, and rounding, of the terms' magnitudes
  const float md = kM * s12;
  float dmin = fdot(nd, g.p0), dmax = dmin;
  {
    const float x = fdot(nd, g.B) * (float)(8 * SW - 1), y = fdot(nd, g.C) * (float)(8 * SH - 1);
    dmin = dmin + (fminf(x, 0.0f) + fminf(y, 0.0f));
    dmax = dmax + (fmaxf(x, 0.0f) + fmaxf(y, 0.0f));
  }
  const bool pos = dmin > md, neg = dmax < -md, sided = pos || neg;
  const float least = pos ? dmin : -dmax;  // of |det|, when sided
  const float sg = neg ? -1.0f : 1.0f;
  bool miss = fmaxf(dmax, -dmin) * 1.1f + md < 0.0001f;  // below mt_isect's least det
  // the greatest value of sg (u det, v det, (1 - u - v) det) over each subtile
  bool cover[SW * SH];
#pragma unroll
  for (int s = 0; s < SW * SH; ++s) cover[s] = on && !miss;
  auto exclude = [&](f3 f, float margin) {
    const float f0 = sg * fdot(f, g.p0), fx = sg * fdot(f, g.B), fy = sg * fdot(f, g.C);
    float mx[SW], my[SH];
#pragma unroll
    for (int i = 0; i < SW; ++i) mx[i] = f0 + fmaxf(fx * (float)(8 * i), fx * (float)(8 * i + 7));
#pragma unroll
    for (int i = 0; i < SH; ++i) my[i] = margin + fmaxf(fy * (float)(8 * i), fy * (float)(8 * i + 7));
#pragma unroll
    for (int s = 0; s < SW * SH; ++s) cover[s] = cover[s] && !(sided && mx[s % SW] + my[s / SW] < 0.0f);
  };
  exclude(nu, kM * su);
  exclude(nv, kM * sv);
  exclude((nd - nu) - nv, kM * (s12 + su + sv));
  // Least distance mt_isect can return for a ray of the block: the nearest
  // vertex along the centre, less the rounding of t, u and v, which a small
  // det magnifies.
  const float da = fmaxf(0.0001f, sided ? 0.93f * least - md : 0.0f);
  const float rda = __builtin_amdgcn_rcpf(da);
  const float key = fminf(0.0f, fminf(fdot(e1, g.c), fdot(e2, g.c))) - fdot(tv, g.c) - 1e-5f * (st + s1 + s2) -
                    2e-5f * (st * s12) * rda;
  bool keep = false;
  unsigned long long cov[SW * SH];
#pragma unroll
  for (int s = 0; s < SW * SH; ++s) {
    cov[s] = __ballot(cover[s]);
    keep = keep || cover[s];
  }
  const unsigned long long kept = __ballot(keep);
  if (!kept) return;
  __syncthreads();  // the batch before has been read
  if (keep) {
    float4* w = L.tri + 4 * lane;
    w[0] = make_float4(nd.x, nd.y, nd.z, key);
    const float mr = 1.5e-6f * (s12 + su + sv);
    w[1] = make_float4(nu.x, nu.y, nu.z, mr);
    w[2] = make_float4(nv.x, nv.y, nv.z, tn);
    w[3] = make_float4(fmaf(2e-6f * s12, rda, 1e-6f), __int_as_float(ent.x), __int_as_float(ent.y), 0.0001f + mr);
  }
  __syncthreads();
  const unsigned long long front = __ballot(keep && pos);
#pragma unroll 1
  for (int pass = 0; pass < 2; ++pass) {
    unsigned long long m = pass ? kept & ~front : front;
    if (!m) continue;
    auto test = [&](const TileTri& w, int i) {
#pragma unroll
      for (int q = 0; q < SW * SH; ++q)
        if ((cov[q] >> i) & 1) test_tri(w, ray[q], o, tris, X);
    };
    // the next triangle is read before the current one is tested
    int i = __builtin_ctzll(m);
    TileTri u = read_tri(L.tri + 4 * i);
    for (;;) {
      m &= m - 1;
      const int j = m ? __builtin_ctzll(m) : i;
      const TileTri v = read_tri(L.tri + 4 * j);
      test(u, i);
      if (!m) break;
      m &= m - 1;
      i = m ? __builtin_ctzll(m) : j;
      u = read_tri(L.tri + 4 * i);
      test(v, j);
      if (!m) break;
    }
  }
}

template <int SW, int SH>
__global__ __launch_bounds__(64, 5) void k_render_block(ffsrl_batch b, ffsrl_camera cam, int env_begin,
                                                     const int32_t* list, int n_env, RenderOut out, int depth) {
  constexpr int NS = SW * SH;
  extern __shared__ int4 tile_lds[];
  const int lane = threadIdx.x;
  const int RW = 2 * cam.width, RH = 2 * cam.height;
  // the XCD-aware mapping of k_render
  const int sub_x = RW >> 3, sub_y = RH >> 3;
  const int blocks_x = (sub_x + SW - 1) / SW, blocks = blocks_x * ((sub_y + SH - 1) / SH);
  const int xcd = blockIdx.x % kXcds, q = blockIdx.x / kXcds;
  const int el = (q / blocks) * kXcds + xcd, blk = q % blocks;
  if (el >= n_env) return;
  const int env = list ? list[el] : env_begin + el;
  const int64_t oi = list ? env : el;  // output slot
  const int x0 = (blk % blocks_x) * SW, y0 = (blk / blocks_x) * SH;
  const int nx = min(SW, sub_x - x0), ny = min(SH, sub_y - y0);  // subtiles inside the image
  const ffsrl_env_desc e = b.envs[env];
  const int64_t vb = e.vbase, sb = e.boundbase, fb = e.fbase;
  const f3 o = mk(cam.origin[0], cam.origin[1], cam.origin[2]);
  const float4* blo = reinterpret_cast<const float4*>(b.bvh_lo) + sb;
  const float4* bhi = reinterpret_cast<const float4*>(b.bvh_hi) + sb;
  const int4* tris = reinterpret_cast<const int4*>(b.tris) + fb;
  const float4* X = reinterpret_cast<const float4*>(b.x) + vb;
  TileLds L;
  L.grid = reinterpret_cast<float4*>(tile_lds);
  L.list = reinterpret_cast<int2*>(tile_lds + 8);
  int* work = reinterpret_cast<int*>(tile_lds) + (kTileGridBytes + kTileListBytes) / 4;
  L.tri = reinterpret_cast<float4*>(work);
  L.stack = work + 64 * 16;
  auto dir = [&](int row, int col) { return xyz(ldu4(reinterpret_cast<const float4*>(cam.dirs), row * RW + col)); };
  const int c0 = 8 * x0, r0 = 8 * y0, c1 = c0 + 8 * nx - 1, r1 = r0 + 8 * ny - 1;
  const int lc = lane & 7, lr = lane >> 3;
  TileRay ray[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s)  // subtiles outside the image repeat its edge
    ray[s] = TileRay{dir(min(r0 + 8 * (s / SW), r1 - 7) + lr, min(c0 + 8 * (s % SW), c1 - 7) + lc), 1e6f, 1e6f, 1e6f,
                     -1, -1};
  const RayGrid g = make_grid(image_axis(dir(0, 0), dir(0, RW - 1), dir(RH - 1, 0), dir(RH - 1, RW - 1)), dir(r0, c0), dir(r0, c1), dir(r1, c0), dir(r1, c1), c1 - c0 + 1, r1 - r0 + 1);
  bool ok = true;
#pragma unroll
  for (int s = 0; s < NS; ++s)
    ok = ok && on_grid(g, ray[s].d, min(8 * (s % SW), c1 - c0 - 7) + lc, min(8 * (s / SW), r1 - r0 - 7) + lr);
  int whole = __all(ok);  // every triangle that a ray can hit is tested
  if (whole) {
    if (lane == 0) put_grid(L.grid, g);
    int ns = 0, nl = 0, steps = 0;
    {
      const float4 lo = ldu4(blo, 0), hi = ldu4(bhi, 0);
      const int outside = box_outside(g, o, lo, hi);
      whole = outside >= 0 && take_nodes(L, 0, lo, hi, lane == 0 && outside == 0, ns, nl);
      __syncthreads();
    }
    whole = __builtin_amdgcn_readfirstlane(whole);
    while (whole && (ns || nl)) {
      while (whole && ns && nl < 64) {
        whole = walk_step(o, blo, bhi, L, ns, nl) && ++steps <= e.nn;
        whole = __builtin_amdgcn_readfirstlane(whole);
        ns = __builtin_amdgcn_readfirstlane(ns);
        nl = __builtin_amdgcn_readfirstlane(nl);
      }
      const int n = nl < 64 ? nl : 64;  // the newest entries: the list shrinks from its end
      if (whole && n) test_batch<SW, SH>(o, tris, X, L, nl - n, n, ray);
      nl -= n;
      __syncthreads();
    }
  }
  const int64_t rays_env = (int64_t)RW * RH;
#pragma unroll 1
  for (int s = 0; s < NS; ++s) {
    if (s % SW >= nx || s / SW >= ny) continue;
    TileRay r = ray[0];
#pragma unroll
    for (int k = 1; k < NS; ++k)
      if (s == k) r = ray[k];
    const f3 d = r.d;
    const int col = c0 + 8 * (s % SW) + lc, row = r0 + 8 * (s / SW) + lr;
    float tMin = 1e6f;
    int best = r.best;
    bool redo = !whole;
    if (__any(best >= 0)) {
      if (!redo && best >= 0) {
        const int4 t = ldu4(tris, best);
        tMin = mt_isect(xyz(ldu4(X, t.x)), xyz(ldu4(X, t.y)), xyz(ldu4(X, t.z)), o, d);
        const f3 lo = xyz(ldu4(blo, r.leaf)), hi = xyz(ldu4(bhi, r.leaf));
        // a zero component with the origin on a face of the leaf or of an
        // ancestor gives NaN slab values; strictly inside the leaf's slab it is
        // inside the ancestors' too
        auto plain = [](float c, float o1, float l1, float h1) {
          return (fabsf(c) >= 1e-30f) | ((c == 0.0f) & (l1 < o1) & (o1 < h1));
        };
        redo = !(tMin > 0.0f && tMin < r.lo2 && plain(d.x, o.x, lo.x, hi.x) && plain(d.y, o.y, lo.y, hi.y) &&
                 plain(d.z, o.z, lo.z, hi.z));
        // the hardware reciprocal (1 ulp) keeps the slab values within 4 ulp of
        // the quotients, half of visit_node's margin
        const f3 inv = mk(__builtin_amdgcn_rcpf(d.x), __builtin_amdgcn_rcpf(d.y), __builtin_amdgcn_rcpf(d.z));
        if (!redo && !visit_node(o, d, inv, lo, hi, tMin, true)) {
          // the box's entry tb is not before t: the leaf is visited all the
          // same if every other distance is beyond tb (triangles left untested
          // are farther than 6e-6 beyond t)
          float tb;
          redo = !(isect_aabb(o, d, lo, hi, &tb) && tb <= tMin * 1.000004f && tb < r.lo2);
        }
      }
    }
    if (__any(redo)) {
      __syncthreads();
      if (redo) {
        const f3 inv = mk(1.0f / d.x, 1.0f / d.y, 1.0f / d.z);
        const RayHit h = trace_ray(blo, bhi, tris, X, o, d, inv, ray_dir_ok(d), work + lane, depth);
        tMin = h.t;
        best = h.best;
      }
      __syncthreads();
    }
    finish_ray(b, cam, out, lane, oi, rays_env, row * RW + col, row, col, vb, fb, o, d, tMin, best);
  }
}

// Area-weighted vertex normals: one thread per vertex sums the area normals
// cross(b - a, c - a) of its faces in increasing face id, then normalizes.
__global__ __launch_bounds__(256) void k_normals(ffsrl_batch b, int env_begin, float* normals) {
  const ffsrl_env_desc e = b.envs[env_begin + blockIdx.y];
  const int v = blockIdx.x * 256 + threadIdx.x;
  if (v >= e.nv) return;
  const int64_t vb = e.vbase;
  const int32_t* off = b.vf_off + e.vtopo_base;
  const int32_t* idx = b.vf_idx + 3 * (int64_t)e.fbase;
  f3 s = mk(0.0f, 0.0f, 0.0f);
  for (int k = off[v]; k < off[v + 1]; ++k) {
    const int4 t = ldi4(b.tris, (int64_t)e.fbase + idx[k]);
    const f3 A = xyz(ld4(b.x, vb + t.x)), B = xyz(ld4(b.x, vb + t.y)), C = xyz(ld4(b.x, vb + t.z));
    s = s + cross(B - A, C - A);
  }
  const f3 n = normalize(s);
  st4(normals, vb + v, make_float4(n.x, n.y, n.z, 0.0f));
}

}  // namespace ffsrl

using namespace ffsrl;

// Block size of the automatic traversal, by the number of 2x2-subtile blocks
// in the launch.  A larger block shares its walk and its triangles' set-up
// among more rays, a smaller one gives more and shorter wavefronts.  Measured
// (us, blocks 1x1 / 2x1 / 2x2): 64x64 depth of the liver scene, 64 envs (4,096
// blocks) 83 / 91 / 105, 256 (16,384) 203 / 166 / 154, 1024 (65,536) 706 / 507 /
// 428; of mixed 1k-40k-tet scenes, 96 (6,144) 95 / 100 / 125, 192 (12,288) 161 /
// 152 / 172, 768 (49,152) 552 / 436 / 419; 128x128 RGB-D of 20k-tet
// ellipsoids, 24 (6,144) 84 / 76 / 77, 384 (98,304) 1048 / 770 / 653.
constexpr int64_t kBlockWide = 5120, kBlockSquare = 16384;

extern "C" {

static int render(const ffsrl_batch* b, const ffsrl_camera* cam, int32_t eb, const int32_t* list, int32_t n,
                  const RenderOut& out, hipStream_t st) {
  if (!b || !cam || !b->envs || !b->x || !b->tris || !b->bvh_lo || !b->bvh_hi || !cam->dirs)
    return fail(FFSRL_E_ARG, "render needs positions, triangles, BVH bounds and ray directions");
  if (cam->width <= 0 || cam->height <= 0 || (cam->width & 3) || (cam->height & 3))
    return fail(FFSRL_E_ARG, "render size %dx%d: width and height must be positive multiples of 4", cam->height,
                cam->width);
  const int m = cam->mode;
  if (m < 0 || m > 5) return fail(FFSRL_E_ARG, "render mode %d", m);
  if (m == 4 && !out.depth && !out.hit) return fail(FFSRL_E_ARG, "depth mode needs a depth (or hit) output");
  // a colour mode also writes the depth image of the same traversal when a
  // depth output is given (RGB-D in one pass)
  if (m != 4 && (!out.rgb || !out.normals)) return fail(FFSRL_E_ARG, "colour modes need rgb output and normals");
  if ((m == 3 || m == 1) && !out.vcolor) return fail(FFSRL_E_ARG, "vertex colour and texture modes need vertex colours");
  if (m == 1 && b->tri_tex && (!b->tri_uv || !b->texels || !b->tex_info))
    return fail(FFSRL_E_ARG, "texture mode: triangle textures given without coordinates, texels or texture table");
  if (m == 5 && !out.tcolor) return fail(FFSRL_E_ARG, "triangle colour mode needs triangle colours");
  if (cam->traversal < 0 || cam->traversal > 2) return fail(FFSRL_E_ARG, "render traversal %d", cam->traversal);
  if (n == 0) return 0;
  const bool quad = cam->traversal == FFSRL_TRAVERSE_QUAD ||
                    (cam->traversal == FFSRL_TRAVERSE_AUTO && cam->width * cam->height >= kQuadMinPixels);
  const int tiles = quad ? ((cam->width + 7) / 8) * ((cam->height + 7) / 8) : (cam->width / 4) * (cam->height / 4);
  // Stack entries per ray: the deepest BVH of the envs (levels = max level + 1
  // bounds the stack of this right-first DFS; a list is bounded by the whole
  // table); kStack without a host mirror.
  int stack_depth = kStack;
  if (b->host_envs) {
    stack_depth = 2;
    const int lo = list ? 0 : eb, hi = list ? b->n_env : eb + n;
    for (int i = lo; i < hi; ++i) {
      stack_depth = std::max(stack_depth, (int)b->host_envs[i].bvh_depth + 1);
      if (quad && b->host_envs[i].nn > kNodeMask)  // a quad stack entry holds a node id in 28 bits
        return fail(FFSRL_E_LIMIT, "env %d: %d BVH nodes exceed the ray stack's %d", i, b->host_envs[i].nn, kNodeMask);
    }
    if (stack_depth > kStack) return fail(FFSRL_E_LIMIT, "BVH with %d levels exceeds the %d-entry ray stack",
                                          stack_depth - 1, kStack);
  }
  if (cam->traversal == FFSRL_TRAVERSE_AUTO) {
    const int sub_x = cam->width / 4, sub_y = cam->height / 4;
    const int64_t groups = (n + kXcds - 1) / kXcds;
    // subtiles per wavefront, by the number of 2x2 blocks in the launch
    const int64_t wide = (int64_t)n * ((sub_x + 1) / 2) * ((sub_y + 1) / 2);
    const int sw = wide < kBlockWide ? 1 : 2, sh = wide < kBlockSquare ? 1 : 2;
    const int64_t blocks = (int64_t)((sub_x + sw - 1) / sw) * ((sub_y + sh - 1) / sh);
    if (groups * kXcds * blocks > INT32_MAX) return fail(FFSRL_E_LIMIT, "render grid too large");
    const int lds = kTileGridBytes + kTileListBytes + std::max(kTileWorkBytes, stack_depth * 64 * (int)sizeof(int));
    auto kern = sh == 2 ? k_render_block<2, 2> : sw == 2 ? k_render_block<2, 1> : k_render_block<1, 1>;
    hipLaunchKernelGGL(kern, dim3((unsigned)(groups * kXcds * blocks)), dim3(64), lds, st, *b, *cam, eb, list, n, out,
                       stack_depth);
    FFSRL_HIP(hipGetLastError());
    return 0;
  }
  const int lds = kWaves * stack_depth * 64 * (int)sizeof(int);
  const int64_t bpe = (tiles + kWaves - 1) / kWaves, groups = (n + kXcds - 1) / kXcds;
  if (groups * kXcds * bpe > INT32_MAX) return fail(FFSRL_E_LIMIT, "render grid too large");
  if (quad)
    hipLaunchKernelGGL(k_render_quad, dim3((unsigned)(groups * kXcds * bpe)), dim3(64 * kWaves), lds, st, *b, *cam,
                       eb, list, n, out, stack_depth);
  else
    hipLaunchKernelGGL(k_render, dim3((unsigned)(groups * kXcds * bpe)), dim3(64 * kWaves), lds, st, *b, *cam, eb,
                       list, n, out, stack_depth);
  FFSRL_HIP(hipGetLastError());
  return 0;
}

int ffsrl_render(const ffsrl_batch* b, const ffsrl_camera* cam, int32_t eb, int32_t ee, float* depth, float* rgb,
                 const float* normals, const float* vcolor, const float* tcolor, int32_t* hit, float* thit,
                 void* stream) {
  if (!b) return fail(FFSRL_E_ARG, "batch NULL");
  if (eb < 0 || ee > b->n_env || eb > ee) return fail(FFSRL_E_ARG, "env range [%d,%d) outside [0,%d)", eb, ee, b->n_env);
  return render(b, cam, eb, nullptr, ee - eb, RenderOut{depth, rgb, normals, vcolor, tcolor, hit, thit},
                as_stream(stream));
}

int ffsrl_render_envs(const ffsrl_batch* b, const ffsrl_camera* cam, const int32_t* envs, int32_t n, float* depth,
                      float* rgb, const float* normals, const float* vcolor, const float* tcolor, int32_t* hit,
                      float* thit, void* stream) {
  if (!b) return fail(FFSRL_E_ARG, "batch NULL");
  if (n < 0 || n > b->n_env || (n > 0 && !envs))
    return fail(FFSRL_E_ARG, "env list of %d entries (batch has %d envs)", n, b->n_env);
  return render(b, cam, 0, envs, n, RenderOut{depth, rgb, normals, vcolor, tcolor, hit, thit}, as_stream(stream));
}

int ffsrl_vertex_normals(const ffsrl_batch* b, int32_t eb, int32_t ee, float* normals, void* stream) {
  if (!b || !b->envs || !b->x || !b->tris || !normals || !b->vf_off || !b->vf_idx)
    return fail(FFSRL_E_ARG, "normals: NULL argument (positions, triangles, vertex-face adjacency, output)");
  if (eb < 0 || ee > b->n_env || eb > ee) return fail(FFSRL_E_ARG, "env range [%d,%d) outside [0,%d)", eb, ee, b->n_env);
  if (ee == eb) return 0;
  if (ee - eb > 65535) return fail(FFSRL_E_LIMIT, "at most 65535 environments per normals call");
  const int nv = b->max_nv < 1 ? 1 : b->max_nv;
  hipLaunchKernelGGL(k_normals, dim3((nv + 255) / 256, ee - eb), dim3(256), 0, as_stream(stream), *b, eb, normals);
  FFSRL_HIP(hipGetLastError());
  return 0;
}

}  // extern "C"
