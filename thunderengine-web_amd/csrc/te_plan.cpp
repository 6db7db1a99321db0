// Which words of the memory a dispatch reads and writes, and which dispatches
// may run side by side (the runtime's batches, te_runtime.hip).
#include <algorithm>
#include <cstring>

#include "te_internal.hpp"

namespace te {

namespace {

// The operands of a kernel that a batch can hold, by parameter.  Every listed
// parameter is one the kernel always uses, so that a parameter at word 0 counts
// like any other; operands that depend on the dispatch are added in op_words.
struct Use {
  std::vector<int> reads, writes;        // fields
  std::vector<int> levels;               // profiles, a word per level
  std::vector<std::pair<int, int>> few;  // parameter words: parameter, words
  bool metric = false;                   // the metric buffer (parameter 30)
};

const std::map<std::string, Use>& uses() {
  static const std::map<std::string, Use> all = [] {
    std::map<std::string, Use> m = {
        {"rayleigh_damping", {{1, 2, 3, 4}, {10, 11, 12, 13}, {5, 6, 7, 8, 19}, {{9, 1}, {16, 1}, {17, 1}}, false}},
        {"turb_rho_faces", {{1}, {4, 5}, {2, 3}, {{6, 3}, {7, 3}}, false}},
        {"turb_def_centers", {{1, 2, 3, 4}, {6, 7, 8, 9}, {5}, {}, true}},
        {"turb_def_faces", {{1, 2, 3, 4}, {6, 7}, {5}, {}, true}},
        {"turb_def_assemble", {{1, 2, 3, 4, 5, 6, 9}, {10, 11}, {7, 8}, {}, false}},
        {"turb_nm", {{1, 2, 5, 6, 7, 8, 9, 10, 11}, {15, 17}, {3, 4, 12, 13, 14}, {{16, 1}, {18, 1}}, false}},
        {"turb_km_kh", {{1, 2, 9}, {4, 5, 6, 7, 8, 9}, {3}, {{10, 1}, {11, 1}, {12, 1}}, true}},
        {"turb_dissipative_heating", {{1, 3, 4, 5, 6, 7, 8, 9, 10}, {10}, {2}, {{11, 5}}, false}},
        {"turb_gettau", {{1, 2, 3, 4, 5, 6, 7, 8}, {3, 4, 5, 6, 7, 8}, {}, {}, false}},
        {"tke_sources", {{1, 2, 3, 4}, {5}, {}, {}, false}},
        {"turb_scalar_flux_h", {{1, 2, 3}, {5, 6}, {}, {{4, 1}}, true}},
        {"tke_flux_h", {{1, 2, 3}, {4, 5}, {}, {}, true}},
        {"turb_openbc_flux", {{1, 2}, {1, 2}, {}, {{3, 2}}, false}},
        {"update_diagnostics_moist",
         {{1, 2, 9, 10, 11, 12, 13, 14}, {15, 16, 17, 18, 19}, {3, 4, 5, 6, 7, 8}, {}, false}},
        {"update_diagnostics", {{1, 2}, {5, 6, 7, 9}, {3, 4, 8}, {}, false}},
        {"stage_tendency_reset", {{}, {1, 2, 3}, {}, {}, false}},
        {"stage_state_reset", {{1, 2, 3, 4, 10}, {5, 6, 7, 8, 9}, {}, {}, false}},
        {"massflux_div", {{1, 2, 3}, {6, 7, 8, 10}, {4, 5, 9}, {}, true}},
        {"build_sadv", {{2}, {3}, {1}, {}, false}},
        {"ppx_finish_xy", {{1, 2}, {2}, {}, {}, false}},
        {"diabatic_rates", {{2, 3, 4, 5, 6, 7, 8, 9}, {6, 7, 8, 9}, {}, {{1, 1}}, false}},
        {"pressure_tendency",
         {{1, 2, 3, 4, 5, 6, 13}, {11}, {7, 8}, {{9, 1}, {10, 1}, {12, 1}, {14, 1}}, false}},
        {"update_rho_prs", {{2, 3, 6}, {7, 8}, {4, 5}, {{1, 1}}, false}},
        {"tke_advance_xy", {{1, 2, 4}, {4}, {}, {{3, 1}}, false}},
        {"rk_update_xy", {{2, 3, 4}, {4}, {}, {{5, 1}}, false}},
        {"tendency_reset_add", {{4, 5, 6}, {1, 2, 3}, {}, {{7, 1}}, false}},
        {"zero_fields", {{}, {}, {}, {{9, 1}}, false}},
        {"copy_fields", {{}, {}, {}, {{9, 1}}, false}},
        {"turb_u_tendency_lds",
         {{1, 2, 3, 4, 5, 6, 7, 8, 14, 15}, {14, 15}, {9, 10}, {{11, 1}, {16, 2}, {17, 1}}, true}},
        {"turb_w_tendency_lds", {{1, 2, 3, 4, 5, 6, 7, 13}, {13}, {8, 9}, {{10, 1}, {14, 2}, {15, 1}}, true}},
        {"turb_scalar_vert_implicit_lds",
         {{1, 2, 3, 4, 5, 8, 9, 13}, {13}, {6, 7}, {{10, 1}, {15, 1}, {16, 1}, {17, 4}, {18, 1}}, true}},
        {"tke_transport_lds", {{1, 2, 3, 4, 5, 11, 12, 13}, {13}, {6, 7}, {{8, 1}, {14, 2}, {15, 1}}, true}},
        {"adv_fused",
         {{2, 4, 6, 13, 14}, {}, {7, 8, 9, 10, 15, 16}, {{1, 1}, {3, 1}, {5, 1}, {12, 1}, {17, 2}, {20, 1}, {21, 1}, {32, 1}},
          true}},
        {"adv_pdef",
         {{2, 4, 6, 13, 14, 43, 44, 46}, {11, 22, 23, 24, 43, 44, 45}, {7, 8, 9, 10, 15, 16},
          {{1, 1}, {3, 1}, {5, 1}, {17, 2}, {20, 1}, {21, 1}, {41, 1}}, true}}};
    m["turb_v_tendency_lds"] = m["turb_u_tendency_lds"];
    m["turb_km_kh_xy"] = m["turb_km_kh"];
    return m;
  }();
  return all;
}

const Use* use_of(int kid) {
  static const std::vector<const Use*> byId = [] {
    std::vector<const Use*> v;
    for (int k = 0; k < te_kernel_count(); ++k) {
      const auto it = uses().find(kernel_name(k));
      v.push_back(it == uses().end() ? nullptr : &it->second);
    }
    return v;
  }();
  return kid >= 0 && kid < (int)byId.size() ? byId[kid] : nullptr;
}

bool meet(const std::vector<Words>& a, const std::vector<Words>& b) {
  for (const Words& x : a)
    for (const Words& y : b)
      if (x.at < y.at + y.n && y.at < x.at + x.n) return true;
  return false;
}

}  // namespace

bool op_words(const Op& op, OpWords& w) {
  w = {};
  const Use* u = use_of(op.kid);
  if (!u) return false;
  const std::string name = kernel_name(op.kid);
  const uint64_t nx = op.nx, ny = op.ny, nz = op.nz, sJ = op.sJ, sK = op.sK;
  // a field: its slot, and the words of its last cell where the strides give more
  const uint64_t plane = std::max(sJ * sK, nx + 7 + sJ * (ny + 6));
  const uint64_t field = std::max(sJ * sK * (nz + 1), nx + 7 + sJ * (ny + 6 + sK * nz));
  const uint64_t level = nz + 1, metric = std::max(2 * (sJ + sK), std::max(sJ + nx + 7, 2 * sJ + sK + ny + 7));
  auto rd = [&](int q, uint64_t n) { w.reads.push_back({op.A[4 + q], n}); };
  auto wr = [&](int q, uint64_t n) { w.writes.push_back({op.A[4 + q], n}); };
  rd(0, 8);
  for (int q : u->reads) rd(q, field);
  for (int q : u->writes) wr(q, field);
  for (int q : u->levels) rd(q, level);
  for (const auto& f : u->few) rd(f.first, (uint64_t)f.second);
  if (u->metric) rd(30, metric);
  // the open sides of a launch that fills halos: none at word 0 (open_sides)
  auto sides = [&](int q) {
    if (op.A[4 + q] != 0) rd(q, 2);
  };
  if (name == "rayleigh_damping") {  // lateral rates along x and y, the means of u, v and theta
    rd(14, nx);
    rd(15, ny);
    rd(18, 3 * nz);
  } else if (name == "turb_dissipative_heating") {  // planes 3 and 4 of the surface buffer
    rd(12, 4 * sJ * sK + plane);
  } else if (name == "turb_scalar_vert_implicit_lds") {  // the surface flux
    rd(14, plane);
  } else if (name == "zero_fields") {
    for (int q = 0; q < std::min(op.count, 8); ++q) wr(1 + q, field);
  } else if (name == "copy_fields") {  // A[0] words each, whatever the grid
    for (int q = 0; q < std::min(op.count, 4); ++q) {
      rd(1 + q, op.A[0]);
      wr(5 + q, op.A[0]);
    }
  } else if (name == "ppx_finish_xy") {
    sides(3);
  } else if (name == "tke_advance_xy") {
    sides(5);
  } else if (name == "rk_update_xy") {
    sides(6);
  } else if (name == "adv_fused") {  // by its chain flags (k_adv.hip)
    if (op.chain & 1) {
      rd(33, field);
      rd(34, field);
    }
    for (int q = 0; q < 2; ++q)
      if (op.chain & (2 << q)) {
        rd(35 + 2 * q, field);
        rd(36 + 2 * q, 1);
      }
    if (op.chain & 64) rd(42, field);
    if (!(op.chain & 16) && op.acc != 0) rd(11, field);
    if (op.chain & 8) {  // the update; the tendency is not stored
      rd(39, field);
      rd(40, field);
      rd(41, 1);
      wr(40, field);
    } else {
      wr(11, field);
    }
  }
  return true;
}

bool independent(const OpWords& a, const OpWords& b) {
  return !meet(a.writes, b.writes) && !meet(a.writes, b.reads) && !meet(a.reads, b.writes);
}

}  // namespace te
