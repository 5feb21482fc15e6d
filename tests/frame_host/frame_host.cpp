// Triangle frames on the host: per (triangle, query) the frame's FP32 squared distance, its error bound
// and w.
#include <algorithm>
using std::max;
using std::min;
#include "../../three-mesh-bvh_amd/csrc/mbvh_frame.h"

extern "C" void frame_distances(const float* tris, const float* queries, int n, float* out) {
  for (int i = 0; i < n; i++) {
    const float *t = tris + 9 * i, *q = queries + 3 * i;
    float4 f[mbvh::kFrameRows];
    mbvh::tri_frame({t[0], t[1], t[2]}, {t[3], t[4], t[5]}, {t[6], t[7], t[8]}, f);
    const float d2 = mbvh::frame_dist2({q[0], q[1], q[2]}, f[0], f[1], f[2], f[3], f[4]);
    out[3 * i] = d2;
    out[3 * i + 1] = mbvh::kFrameRel * d2 + std::fabs(f[0].w);
    out[3 * i + 2] = f[0].w;
  }
}
