// gp_order.h -- the advance's workgroup order in the reference's cell order (x
// fastest, then y, then z): the particles of a z layer are cut into eight y
// blocks, one for each XCD, and every XCD goes through its own y block layer
// by layer.  Layers are taken as equally full (the order is a permutation of
// the workgroups whatever the particles do; how well the caches do depends on
// it).
#pragma once

#include <hip/hip_runtime.h>

namespace gp {

struct LayerMap {
  int nb = 0;       // workgroups with work
  int layers = 0;   // z layers of cells; 0: the plain order
  int per = 0;      // workgroups launched for each (layer, y block), nb's share rounded up
};

// y blocks per XCD where a layer's y block fills four workgroups or more and
// a cell holds fewer than six particles on average.  Advance alone, in us,
// plain order -> y blocks, workgroups a y block and particles a cell in
// brackets:
//   FP32  1e6 on 256^3 (2.5, 0.14) 322 -> 323, 2e6 (4.0, 0.14) 480 -> 472, 4e6
//         (6.3, 0.14) 852 -> 837, 8e6 on 512^3 (12, 0.25) 2528 -> 2329
//   FP64  4e6 on 256^3 1476 -> 1373 (four points 1907 -> 1729), 8e6 on 512^3
//         4367 -> 4138 (5807 -> 5298)
//   fuller cells, FP32: 1e6 (6.6, 2.5) 282 -> 274, (8.4, 5.1) 323 -> 318, (11,
//         13) 359 -> 383; 6e5 (7.2, 8.7) 234 -> 262; 5e5 (7.2, 13) 175 -> 206;
//         2e6 (18, 13) 917 -> 938, FP64 1444 -> 1421
inline LayerMap layer_map(int nb, int np, int nbox, int nz) {
  LayerMap lm;
  if (nb < 32ll * nz || np >= 6ll * nbox) return lm;
  lm.nb = nb;
  lm.layers = nz;
  lm.per = (int)((nb + 8ll * nz - 1) / (8ll * nz));
  return lm;
}
inline int layer_grid(const LayerMap& lm) { return 8 * lm.layers * lm.per; }

// the workgroup of work that block b takes; lm.nb: none
__host__ __device__ __forceinline__ int layer_item(const LayerMap& lm, int b) {
  const int y = b & 7, t = b >> 3, j = t % lm.per, z = t / lm.per;
  const long long k = 8ll * z + y, n = 8ll * lm.layers;
  const int lo = (int)(k * lm.nb / n), hi = (int)((k + 1) * lm.nb / n);
  return lo + j < hi ? lo + j : lm.nb;
}

}  // namespace gp
