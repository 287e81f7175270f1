// Point location in a tetrahedral field by the product's own lists, one entry
// after the other -- test infrastructure.  Built from csrc/tet_grid.h, so the
// lists are those that the GPU searches; without the face planes that rule
// entries out there, the first entry that the containment test accepts is the
// answer by definition, and the GPU's must equal it bit for bit.
#include <cfloat>
#include <cmath>
#include <cstdint>

#include "../anari-visionaray_amd/csrc/tet_grid.h"

namespace {

struct V {
  float x, y, z;
};
V operator-(V a, V b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
float dot(V a, V b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
V cross(V a, V b) {
  return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}

// intersectTet (Plane.h:56-96)
float plane_ratio(V a, V b, V c, V opp) {
  const V n = cross(b - a, c - a);
  const float d = dot(a, n);
  return (dot(V{0.f, 0.f, 0.f}, n) - d) / (dot(opp, n) - d);
}

bool tet_value(V P, const vrt::tetgrid::Rec &r, float &value) {
  V v[4];
  for (int k = 0; k < 4; ++k) v[k] = V{r.v[k][0], r.v[k][1], r.v[k][2]} - P;
  const float fa = plane_ratio(v[1], v[3], v[2], v[0]);
  if (fa < 0.f || fa > 1.f) return false;
  const float fb = plane_ratio(v[0], v[2], v[3], v[1]);
  if (fb < 0.f) return false;
  const float fc = plane_ratio(v[0], v[3], v[1], v[2]);
  if (fc < 0.f) return false;
  const float fd = plane_ratio(v[0], v[1], v[2], v[3]);
  if (fd < 0.f) return false;
  value = fa * r.v[0][3] + fb * r.v[1][3] + fc * r.v[2][3] + fd * r.v[3][3];
  return true;
}

}  // namespace

// values[i]: the field at pts[i], NaN where no tetrahedron contains it;
// returns the longest list
extern "C" __attribute__((visibility("default"))) int orc_tet_walk(
    const float *pos, const float *vdata, const uint32_t *index, int64_t num_tets, int n,
    const float *pts, float *values) {
  using namespace vrt::tetgrid;
  std::vector<Rec> recs(static_cast<size_t>(num_tets));
  float lo[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, hi[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
  for (size_t t = 0; t < recs.size(); ++t)
    for (int k = 0; k < 4; ++k) {
      const size_t i = index[4 * t + k];
      for (int a = 0; a < 3; ++a) {
        recs[t].v[k][a] = pos[3 * i + a];
        lo[a] = std::fmin(lo[a], pos[3 * i + a]);
        hi[a] = std::fmax(hi[a], pos[3 * i + a]);
      }
      recs[t].v[k][3] = vdata[i];
    }
  Grid g;
  if (!build(recs, lo, hi, 1.0, 0, g)) return -1;
  parallel_for(size_t(n), 0, [&](size_t p) {
    const V P{pts[3 * p], pts[3 * p + 1], pts[3 * p + 2]};
    values[p] = NAN;
    if (!(P.x >= lo[0] && P.x <= hi[0] && P.y >= lo[1] && P.y <= hi[1] && P.z >= lo[2] &&
          P.z <= hi[2]))
      return;
    const float q[3] = {(P.x - g.lo[0]) * g.inv_cell[0], (P.y - g.lo[1]) * g.inv_cell[1],
                        (P.z - g.lo[2]) * g.inv_cell[2]};
    size_t c[3];
    for (int a = 0; a < 3; ++a) c[a] = std::min(uint32_t(q[a]), uint32_t(g.dims[a] - 1));
    const size_t cell = (c[2] * g.dims[1] + c[1]) * g.dims[0] + c[0];
    for (uint32_t i = g.start[cell]; i < g.start[cell + 1]; ++i) {
      float v;
      if (tet_value(P, g.recs[i], v)) {
        values[p] = v;
        return;
      }
    }
  });
  return int(g.max_list);
}
