// Phases P4 (islands: union-find over the dynamic pairs, sleep, the island sort of the active manifolds) and P5 (the
// sequential-impulse solver: contact and friction rows, special synthetic rows for the ball's static contacts, 10 split-impulse
// iterations, up to 10 velocity iterations with a zero-residual exit, finish). Reference: cuda/sim/simulation_island_manager.cuh,
// seq_impulse_constraint_solver.cuh, solver_constraint.cuh.
#pragma once
#include "rs_narrow.h"

namespace rs {

// ---- P4 ----------------------------------------------------------------------------------------------------------------------
RS_FN int island_root(int* parent, int i) {  // find with full path compression (:29-39)
  int r = i;
  while (parent[r] != r) r = parent[r];
  while (parent[i] != r && i != r) {
    int nx = parent[i];
    parent[i] = r;
    i = nx;
  }
  return r;
}
// Up to 16 values of 4 bits (the active list: manifold indices) in one register: an index into it is a shift.
struct Nibbles {
  uint64_t v;
  RS_FN uint32_t get(int i) const { return (uint32_t)(v >> (4 * i)) & 15u; }
  RS_FN void set(int i, uint32_t x) { v = (v & ~(15ull << (4 * i))) | ((uint64_t)x << (4 * i)); }
};
// Hoare partition sort of idx[0..n-1] by the keys of its values (key m: bits 2m, 2m + 1 of keys) (:43-66, the recursive
// form's visiting order on an explicit stack). The ranges on the stack are disjoint and hold two entries or more, so at
// most eight of them, packed as the two nibbles of a byte each.
RS_FN void hoare_sort(Nibbles& idx, int n, uint32_t keys) {
  if (n <= 1) return;
  uint64_t stack = (uint64_t)(n - 1) << 4;
  int sp = 1;
  while (sp > 0) {
    --sp;
    const uint32_t range = (uint32_t)(stack >> (8 * sp)) & 255u;
    int lo = (int)(range & 15u), hi = (int)(range >> 4), i = lo, j = hi;
    const uint32_t pivot = (keys >> (2u * idx.get((lo + hi) / 2))) & 3u;
    for (;;) {
      uint32_t at_i = idx.get(i), at_j = idx.get(j);
      while (((keys >> (2u * at_i)) & 3u) < pivot) at_i = idx.get(++i);
      while (pivot < ((keys >> (2u * at_j)) & 3u)) at_j = idx.get(--j);
      if (i > j) break;
      idx.set(i, at_j);
      idx.set(j, at_i);
      ++i;
      if (j == 0) break;
      --j;
      if (i > j) break;
    }
    stack &= sp ? ~0ull >> (64 - 8 * sp) : 0ull;
    if (i < hi) stack |= (uint64_t)((uint32_t)i | (uint32_t)hi << 4) << (8 * sp++);
    if (lo < j) stack |= (uint64_t)((uint32_t)lo | (uint32_t)j << 4) << (8 * sp++);
  }
}
// idx = the n values of v in ascending order (the insertion sort's order; the values are distinct but for a malformed state).
RS_FN Nibbles sorted_nibbles(const uint32_t* v, int n) {
  uint32_t mask = 0;
  RS_UNROLL
  for (int i = 0; i < 16; ++i)
    if (i < n) mask |= 1u << (v[i] & 15u);
  Nibbles idx = {0};
  int at = 0;
  for (uint32_t m = mask; m != 0; m &= m - 1) idx.set(at++, (uint32_t)__builtin_ctz(m));
  if (at == n) return idx;
  idx.v = 0;
  at = 0;
  for (uint32_t x = 0; x < 16; ++x)
    for (int i = 0; i < n; ++i)
      if ((v[i] & 15u) == x) idx.set(at++, x);
  return idx;
}
// The pairs, the active list and the manifolds' bodies are read for all their slots at once, and the active list is sorted
// in a register (65,536 contact arenas: 46 -> 27 thousand cycles of a wave's tick; each list entry had been a read that
// waited on the one before, each sort step a private-memory round trip).
RS_INLINE void phase_p4(ArenaState& s, const StaticData& w) {  // :100-150
  static_assert(MAX_MANIFOLDS == 16 && MAX_ACTIVE == 16 && NUM_DYN == 3, "four bits per index, two per key");
  const int n = (int)(s.n_active < (uint32_t)MAX_ACTIVE ? s.n_active : (uint32_t)MAX_ACTIVE);
  const uint32_t np = s.n_pairs < (uint32_t)MAX_PAIRS ? s.n_pairs : (uint32_t)MAX_PAIRS;
  uint32_t activation[NUM_DYN], active[MAX_ACTIVE];
  Pair pairs[MAX_PAIRS];
  RS_UNROLL
  for (int d = 0; d < NUM_DYN; ++d) activation[d] = s.bodies[d].activation;
  RS_UNROLL
  for (int p = 0; p < MAX_PAIRS; ++p) pairs[p] = (uint32_t)p < np ? s.pairs[p] : Pair{0, 0};
  RS_UNROLL
  for (int i = 0; i < MAX_ACTIVE; ++i) active[i] = s.active[i];
  uint32_t moving = 0;  // bit p: neither proxy of pair p is static
  RS_UNROLL
  for (int p = 0; p < MAX_PAIRS; ++p)
    moving |= (uint32_t)((uint32_t)p < np && (w.proxies[pairs[p].proxy0].filter_group & k::FILTER_STATIC) == 0 &&
                         (w.proxies[pairs[p].proxy1].filter_group & k::FILTER_STATIC) == 0) << p;
  int tag[NUM_DYN] = {0, 1, 2};
  if (moving != 0) {
    int parent[NUM_DYN] = {0, 1, 2};
    for (; moving != 0; moving &= moving - 1) {
      const Pair pr = s.pairs[__builtin_ctz(moving)];
      int a = dyn_slot(w, w.proxies[pr.proxy0].client_body), b = dyn_slot(w, w.proxies[pr.proxy1].client_body);
      if (a < 0 || b < 0) continue;
      if ((s.bodies[a].collision_flags & k::CF_NO_CONTACT_RESPONSE) || (s.bodies[b].collision_flags & k::CF_NO_CONTACT_RESPONSE)) continue;
      int r0 = island_root(parent, a), r1 = island_root(parent, b);
      if (r0 != r1) parent[r0] = r1;
    }
    for (int d = 0; d < NUM_DYN; ++d) tag[d] = island_root(parent, d);
  }
  uint32_t awake = 0;  // by tag
  RS_UNROLL
  for (int d = 0; d < NUM_DYN; ++d) awake |= activation[d] == k::ACT_ACTIVE ? 1u << tag[d] : 0u;
  RS_UNROLL
  for (int d = 0; d < NUM_DYN; ++d)
    if (!((awake >> tag[d]) & 1u) && activation[d] == k::ACT_WANTS_DEACTIVATION) body_sleep(s.bodies[d]);
  if (n <= 1) return;
  // a manifold's key: the island tag of its first dynamic body, one up (0 for none)
  uint32_t keys = 0;
  RS_UNROLL
  for (int m = 0; m < MAX_MANIFOLDS; ++m) {
    const int d0 = dyn_slot(w, s.manifolds[m].body0), d1 = dyn_slot(w, s.manifolds[m].body1), d = d0 >= 0 ? d0 : d1;
    const int t = d < 0 ? -1 : d == 0 ? tag[0] : d == 1 ? tag[1] : tag[2];
    keys |= (uint32_t)(t + 1) << (2 * m);
  }
  Nibbles idx = sorted_nibbles(active, n);
  hoare_sort(idx, n, keys);
  RS_UNROLL
  for (int i = 0; i < MAX_ACTIVE; ++i)
    if (i < n) s.active[i] = idx.get(i);
}

// ---- P5 rows (solver_constraint.cuh) -----------------------------------------------------------------------------------------
constexpr int MAX_ROWS = 32;
// The solver bodies: one per dynamic body, at its slot of the state, and the fixed one.
constexpr int FIXED_BODY = NUM_DYN, MAX_SOLVER_BODIES = NUM_DYN + 1;
constexpr int SOLVER_ITERATIONS = 10;
constexpr float ERP2 = 0.8f;
constexpr float SPLIT_TURN_ERP = 0.1f;

struct Row {
  V3 r1xn, n1, r2xn, n2, ang_a, ang_b;
  float applied_push, applied, friction, jinv, rhs, lower, upper, rhs_pen;
  int friction_idx, a, b, split_only;
};
struct RowPoint { V3 normal; float friction, restitution, distance; };
// What the rows read of a body: of a dynamic one its velocities, the accumulated ones and its inertia; a fixed one is zero.
struct SolverSide {
  bool dynamic;
  V3 lin, ang, ext_force, ext_torque;
  M3 inv_inertia;
  float inv_mass;
  V3 pos;
};
RS_FN SolverSide side_fixed() {
  V3 z = splat(0.0f);
  return SolverSide{false, z, z, z, z, M3{z, z, z}, 0.0f, z};
}
RS_FN SolverSide side_of(const Body& b, const BodyConst& c) {
  return SolverSide{true, b.lin_vel, b.ang_vel, b.accum_lin_vel, b.accum_ang_vel, b.inv_inertia_world, c.inv_mass, b.world.t};
}
// The side of dynamic slot d (-1: the fixed one) out of the three held in registers.
RS_FN SolverSide pick_side(const SolverSide* sides, int d) {
  SolverSide v = side_fixed();
  RS_UNROLL
  for (int e = 0; e < NUM_DYN; ++e)
    if (d == e) v = sides[e];
  return v;
}
RS_FN V3 side_vel(const SolverSide& b, V3 rel) { return b.lin + b.ext_force + cross(b.ang + b.ext_torque, rel); }
RS_FN float bullet_dot(V3 a, V3 b) {  // x + (y + z)
  V3 r = a * b;
  return r.x + (r.y + r.z);
}
RS_FN V3 plane_space(V3 n) {  // util.rs plane_space_1
  if (fabs_(n.z) > 0.70710678118654752440f) {
    float kk = 1.0f / __builtin_sqrtf(n.y * n.y + n.z * n.z);
    return V3{0.0f, fneg(n.z) * kk, n.y * kk};
  }
  float kk = 1.0f / __builtin_sqrtf(n.x * n.x + n.y * n.y);
  return V3{fneg(n.y) * kk, n.x * kk, 0.0f};
}
RS_FN V3 lat_friction_dir(const RowPoint& cp, const SolverSide& a, const SolverSide& b, V3 r1, V3 r2) {
  V3 v = side_vel(a, r1) - side_vel(b, r2);
  float rv = dot(cp.normal, v);
  V3 lat = v - cp.normal * rv;
  float l2 = length_sq(lat);
  if (l2 > 1.1920929e-7f) return lat * (1.0f / __builtin_sqrtf(l2));
  return plane_space(cp.normal);
}
RS_FN Row row_new(int a, int b, int fidx, float friction, float lower, float upper) {
  Row r;
  V3 z = splat(0.0f);
  r.r1xn = r.n1 = r.r2xn = r.n2 = r.ang_a = r.ang_b = z;
  r.applied_push = r.applied = r.jinv = r.rhs = r.rhs_pen = 0.0f;
  r.friction = friction;
  r.lower = lower;
  r.upper = upper;
  r.friction_idx = fidx;
  r.a = a;
  r.b = b;
  r.split_only = 0;
  return r;
}
RS_FN Row contact_row(int ia, int ib, const SolverSide& s0, const SolverSide& s1, V3 r1, V3 r2, const RowPoint& cp, int fidx,
                      float dt) {  // get_contact_constraint (warm start is the identity: :205-214)
  Row r = row_new(ia, ib, fidx, cp.friction, 0.0f, 1e10f);
  float inv_dt = 1.0f / dt;
  V3 n = cp.normal;
  float den0 = 0.0f, v1n = 0.0f, den1 = 0.0f, v2n = 0.0f;
  V3 vel0 = splat(0.0f), vel1 = splat(0.0f);
  if (s0.dynamic) {
    V3 ta = cross(r1, n);
    r.ang_a = mul_t(s0.inv_inertia, ta);
    den0 = s0.inv_mass + dot(n, cross(r.ang_a, r1));
    vel0 = s0.lin + cross(s0.ang, r1);
    r.n1 = n;
    r.r1xn = ta;
    v1n = dot(r.n1, s0.lin + s0.ext_force) + dot(r.r1xn, s0.ang + s0.ext_torque);
  }
  if (s1.dynamic) {
    V3 ta = cross(r2, n);
    r.ang_b = mul_t(s1.inv_inertia, -ta);
    den1 = s1.inv_mass + dot(n, cross(-r.ang_b, r2));
    vel1 = s1.lin + cross(s1.ang, r2);
    r.n2 = -n;
    r.r2xn = -ta;
    v2n = dot(r.n2, s1.lin + s1.ext_force) + dot(r.r2xn, s1.ang + s1.ext_torque);
  }
  r.jinv = 1.0f / (den0 + den1);
  float rel_vel = dot(n, vel0 - vel1);
  float restitution = fmax_rs(cp.restitution * fneg(rel_vel), 0.0f);
  float pen = cp.distance;
  float pos_err = pen > 0.0f ? 0.0f : (fneg(pen) * ERP2) * inv_dt;
  float vel_err = restitution - (v1n + v2n);
  float pen_imp = pos_err * r.jinv, vel_imp = vel_err * r.jinv;
  if (pen > 1e30f) {  // SPLIT_IMPULSE_PENETRATION_THRESHOLD
    r.rhs = pen_imp + vel_imp;
    r.rhs_pen = 0.0f;
  } else {
    r.rhs = vel_imp;
    r.rhs_pen = pen_imp;
  }
  return r;
}
RS_FN Row split_only_row(int ia, int ib, const SolverSide& s0, const SolverSide& s1, V3 r1, V3 r2, const RowPoint& cp, float dt) {  // :100-172
  Row r = row_new(ia, ib, -1, cp.friction, 0.0f, 1e10f);
  r.split_only = 1;
  V3 n = cp.normal;
  float den0 = 0.0f, den1 = 0.0f;
  if (s0.dynamic) {
    V3 ta = cross(r1, n);
    r.ang_a = mul_t(s0.inv_inertia, ta);
    den0 = s0.inv_mass + dot(n, cross(r.ang_a, r1));
    r.n1 = n;
    r.r1xn = ta;
  }
  if (s1.dynamic) {
    V3 ta = cross(r2, n);
    r.ang_b = mul_t(s1.inv_inertia, -ta);
    den1 = s1.inv_mass + dot(n, cross(-r.ang_b, r2));
    r.n2 = -n;
    r.r2xn = -ta;
  }
  r.jinv = 1.0f / (den0 + den1);
  float inv_dt = 1.0f / dt, pen = cp.distance;
  float pos_err = pen > 0.0f ? 0.0f : (fneg(pen) * ERP2) * inv_dt;
  float pen_imp = pos_err * r.jinv;
  r.rhs_pen = pen > 1e30f ? 0.0f : pen_imp;
  return r;
}
RS_FN Row friction_row(int ia, int ib, const SolverSide& s0, const SolverSide& s1, V3 r1, V3 r2, float friction, V3 axis, int fidx) {  // get_friction_constraint (:39-67, :291-340)
  Row r = row_new(ia, ib, fidx, friction, fneg(friction), friction);
  float v1n = 0.0f, den1 = 0.0f, v2n = 0.0f, den2 = 0.0f;
  if (s0.dynamic) {
    r.n1 = axis;
    r.r1xn = cross(r1, r.n1);
    r.ang_a = mul_t(s0.inv_inertia, r.r1xn);
    den1 = s0.inv_mass + dot(axis, cross(r.ang_a, r1));
    v1n = dot(r.n1, s0.lin + s0.ext_force) + dot(r.r1xn, s0.ang);
  }
  if (s1.dynamic) {
    r.n2 = -axis;
    r.r2xn = cross(r2, r.n2);
    r.ang_b = mul_t(s1.inv_inertia, r.r2xn);
    den2 = s1.inv_mass + dot(axis, cross(-r.ang_b, r2));
    v2n = dot(r.n2, s1.lin + s1.ext_force) + dot(r.r2xn, s1.ang);
  }
  r.jinv = 1.0f / (den1 + den2);
  r.rhs = fneg(v1n + v2n) * r.jinv;
  return r;
}
// The row solves read and write the bodies' deltas through the bank (fields: 0 dlin, 1 dang, 2 push, 3 turn).
enum BankField { BF_DLIN = 0, BF_DANG = 1, BF_PUSH = 2, BF_TURN = 3, BF_INV_MASS = 4 };
// The row solves read the bodies' inverse masses and kinds from the bank (a body that is not dynamic takes no delta).
RS_FN float resolve_split(Row& r, DeltaBank& bank) {  // :518-565
  if (r.rhs_pen == 0.0f) return 0.0f;
  const bool ha = bank.dynamic(r.a), hb = bank.dynamic(r.b);
  float di = r.rhs_pen;
  V3 pa = ha ? bank.get(r.a, BF_PUSH) : splat(0.0f), ta = ha ? bank.get(r.a, BF_TURN) : splat(0.0f);
  V3 pb = hb ? bank.get(r.b, BF_PUSH) : splat(0.0f), tb = hb ? bank.get(r.b, BF_TURN) : splat(0.0f);
  float d1 = ha ? bullet_dot(r.n1, pa) + bullet_dot(r.r1xn, ta) : 0.0f;
  float d2 = hb ? bullet_dot(r.n2, pb) + bullet_dot(r.r2xn, tb) : 0.0f;
  di = di - d1 * r.jinv;
  di = di - d2 * r.jinv;
  float sum = r.applied_push + di;
  if (sum < r.lower) {
    di = r.lower - r.applied_push;
    r.applied_push = r.lower;
  } else {
    r.applied_push = sum;
  }
  if (ha) {
    bank.set(r.a, BF_PUSH, pa + r.n1 * bank.get(r.a, BF_INV_MASS) * di);
    bank.set(r.a, BF_TURN, ta + r.ang_a * di);
  }
  if (hb) {  // re-read: a and b may be the same body
    bank.set(r.b, BF_PUSH, bank.get(r.b, BF_PUSH) + r.n2 * bank.get(r.b, BF_INV_MASS) * di);
    bank.set(r.b, BF_TURN, bank.get(r.b, BF_TURN) + r.ang_b * di);
  }
  return di / r.jinv;
}
RS_FN float resolve_row(Row& r, DeltaBank& bank, bool two_sided) {  // :427-516
  const bool ha = bank.dynamic(r.a), hb = bank.dynamic(r.b);
  float di = r.rhs;
  V3 la = ha ? bank.get(r.a, BF_DLIN) : splat(0.0f), aa = ha ? bank.get(r.a, BF_DANG) : splat(0.0f);
  V3 lb = hb ? bank.get(r.b, BF_DLIN) : splat(0.0f), ab = hb ? bank.get(r.b, BF_DANG) : splat(0.0f);
  float d1 = ha ? bullet_dot(r.n1, la) + bullet_dot(r.r1xn, aa) : 0.0f;
  float d2 = hb ? bullet_dot(r.n2, lb) + bullet_dot(r.r2xn, ab) : 0.0f;
  di = di - d1 * r.jinv;
  di = di - d2 * r.jinv;
  float sum = r.applied + di;
  if (sum < r.lower) {
    di = r.lower - r.applied;
    r.applied = r.lower;
  } else if (two_sided && sum > r.upper) {
    di = r.upper - r.applied;
    r.applied = r.upper;
  } else {
    r.applied = sum;
  }
  if (ha) {
    bank.set(r.a, BF_DLIN, la + r.n1 * bank.get(r.a, BF_INV_MASS) * di);
    bank.set(r.a, BF_DANG, aa + r.ang_a * di);
  }
  if (hb) {  // re-read: a and b may be the same body
    bank.set(r.b, BF_DLIN, bank.get(r.b, BF_DLIN) + r.n2 * bank.get(r.b, BF_INV_MASS) * di);
    bank.set(r.b, BF_DANG, bank.get(r.b, BF_DANG) + r.ang_b * di);
  }
  return di / r.jinv;
}

// ---- P5 (seq_impulse_constraint_solver.cuh) -----------------------------------------------------------------------------------
struct SpecialAcc {
  V3 normal;
  float lever, friction, restitution;
  uint32_t count;
};
struct Solver {
  Row contact[MAX_ROWS];
  Row friction[MAX_ROWS];
  int n_contact, n_friction;
  uint32_t used;                 // bit d: dynamic body d takes part
  SpecialAcc special[NUM_DYN];   // by dynamic body
  uint32_t special_order;        // the bodies with special contacts in order of their first one, two bits each
  int n_special;
};
RS_FN void add_special(Solver& sv, int d, V3 normal, float lever, float friction, float restitution) {  // :84-99
  RS_UNROLL
  for (int e = 0; e < NUM_DYN; ++e) {
    if (d != e) continue;
    SpecialAcc& a = sv.special[e];
    if (a.count != 0) {
      a.normal += normal;
      a.lever = a.lever + lever;
      a.friction = a.friction + friction;
      a.restitution = a.restitution + restitution;
      a.count += 1;
    } else {
      a = SpecialAcc{normal, lever, friction, restitution, 1u};
      sv.special_order |= (uint32_t)e << (2 * sv.n_special);
      sv.n_special += 1;
    }
  }
}
RS_FN void push_special(Solver& sv, ArenaState& s, const SolverSide& s0, int d, const SpecialAcc& acc, float dt) {  // :102-129
  float ns = (float)acc.count;
  V3 mn = normalize_or_zero(acc.normal / ns);
  float lever = acc.lever / ns, fr = acc.friction / ns, rest = acc.restitution / ns;
  const SolverSide s1 = side_fixed();
  V3 r1 = mn * fneg(lever), r2 = splat(0.0f);
  RowPoint cp = RowPoint{mn, fr, rest, 0.0f};
  int fidx = sv.n_contact;
  if (sv.n_contact >= MAX_ROWS || sv.n_friction >= MAX_ROWS) {
    s.overflow[OVF_ACTIVE]++;
    return;
  }
  sv.contact[sv.n_contact++] = contact_row(d, FIXED_BODY, s0, s1, r1, r2, cp, fidx, dt);
  V3 lat = lat_friction_dir(cp, s0, s1, r1, r2);
  sv.friction[sv.n_friction++] = friction_row(d, FIXED_BODY, s0, s1, r1, r2, cp.friction, lat, fidx);
}
// The three dynamic bodies are read once and picked from registers per manifold; the active list is read at once.
RS_FN void solver_setup(Solver& sv, ArenaState& s, const StaticData& w, float dt) {  // :132-193
  sv.used = 0;
  SolverSide sides[NUM_DYN];
  uint32_t active[MAX_ACTIVE];
  RS_UNROLL
  for (int d = 0; d < NUM_DYN; ++d) {  // setup_solver_bodies
    sides[d] = side_of(s.bodies[d], w.bodies[w.dyn_body[d]]);
    sv.used |= body_active(s.bodies[d]) ? 1u << d : 0u;
    sv.special[d] = SpecialAcc{splat(0.0f), 0.0f, 0.0f, 0.0f, 0u};
  }
  sv.n_special = 0;
  sv.special_order = 0;
  uint64_t list = 0;  // the active manifolds, four bits each
  const uint32_t n = s.n_active < (uint32_t)MAX_ACTIVE ? s.n_active : (uint32_t)MAX_ACTIVE;
  RS_UNROLL
  for (int i = 0; i < MAX_ACTIVE; ++i) active[i] = s.active[i];
  RS_UNROLL
  for (int i = 0; i < MAX_ACTIVE; ++i) list |= (uint64_t)(active[i] & 15u) << (4 * i);
  for (uint32_t ai = 0; ai < n; ++ai) {
    const Manifold& m = s.manifolds[(uint32_t)(list >> (4 * ai)) & 15u];
    int d0 = dyn_slot(w, m.body0), d1 = dyn_slot(w, m.body1);
    const int ia = d0 >= 0 ? d0 : FIXED_BODY, ib = d1 >= 0 ? d1 : FIXED_BODY;
    sv.used |= (d0 >= 0 ? 1u << d0 : 0u) | (d1 >= 0 ? 1u << d1 : 0u);
    const SolverSide s0 = pick_side(sides, d0), s1 = pick_side(sides, d1);
    const V3 p0 = w.bodies[m.body0].pose.t, p1 = w.bodies[m.body1].pose.t;
    V3 t0 = d0 >= 0 ? s0.pos : p0;
    V3 t1 = d1 >= 0 ? s1.pos : p1;
    for (uint32_t pi = 0; pi < m.n_points; ++pi) {
      const ManifoldPoint& mp = m.pts[pi];
      V3 r1 = mp.world_on_a - t0, r2 = mp.world_on_b - t1;
      RowPoint cp = RowPoint{mp.normal_on_b, mp.friction, mp.restitution, mp.distance};
      if (mp.is_special) {
        if (sv.n_contact >= MAX_ROWS) s.overflow[OVF_ACTIVE]++;
        else sv.contact[sv.n_contact++] = split_only_row(ia, ib, s0, s1, r1, r2, cp, dt);
        int obj = -1;
        V3 lever = splat(0.0f);
        if (d0 >= 0) {
          obj = d0;
          lever = r1;
        } else if (d1 >= 0) {
          obj = d1;
          lever = r2;
        }
        if (obj >= 0) add_special(sv, obj, cp.normal, length(lever), cp.friction, cp.restitution);
        continue;
      }
      int fidx = sv.n_contact;
      V3 lat = lat_friction_dir(cp, s0, s1, r1, r2);
      if (sv.n_contact >= MAX_ROWS || sv.n_friction >= MAX_ROWS) {
        s.overflow[OVF_ACTIVE]++;
        continue;
      }
      sv.contact[sv.n_contact++] = contact_row(ia, ib, s0, s1, r1, r2, cp, fidx, dt);
      sv.friction[sv.n_friction++] = friction_row(ia, ib, s0, s1, r1, r2, cp.friction, lat, fidx);
    }
  }
  s.n_active = 0;
  for (int i = 0; i < MAX_ACTIVE; ++i) s.active[i] = 0;
  for (int i = 0; i < sv.n_special; ++i) {
    const int d = (int)((sv.special_order >> (2 * i)) & 3u);
    SpecialAcc acc = sv.special[0];
    RS_UNROLL
    for (int e = 1; e < NUM_DYN; ++e)
      if (d == e) acc = sv.special[e];
    push_special(sv, s, pick_side(sides, d), d, acc, dt);
  }
}
// The iterations (:196-251), the running rows a bit mask, the contact impulses a friction row needs in the bank. The first
// HELD_ROWS rows of each kind, all that most arenas have, are read once and held in registers through the iterations; the
// loops over the rows past them read their next row while they solve the current one (a row's solve never writes another
// row) and write back what a solve changes. Nothing reads a row after the iterations. (65,536 contact arenas: P5 195 -> 152
// thousand cycles of a wave's tick with the rows held, 111 with the bodies held too, see solver_setup. Four rows of each
// kind fill the wave's accumulation registers.)
constexpr int HELD_ROWS = 4;
RS_FN void solver_iterate(Solver& sv, const StaticData& w, DeltaBank& bank) {  // :196-251
  static_assert(MAX_ROWS <= BANK_ROWS && MAX_SOLVER_BODIES == BANK_BODIES, "the bank holds every row and body");
  static_assert(MAX_ROWS <= 32, "the running rows are a 32-bit mask");
  RS_UNROLL
  for (int i = 0; i < MAX_SOLVER_BODIES; ++i) {
    RS_UNROLL
    for (int f = BF_DLIN; f <= BF_TURN; ++f) bank.set(i, f, splat(0.0f));
    bank.set(i, BF_INV_MASS, i < NUM_DYN ? w.bodies[w.dyn_body[i]].inv_mass_splat : splat(0.0f));
    bank.set_dynamic(i, i < NUM_DYN);
  }
  const int nc = sv.n_contact, nf = sv.n_friction;
  Row ch[HELD_ROWS], fh[HELD_ROWS];
  RS_UNROLL
  for (int i = 0; i < HELD_ROWS; ++i) {
    ch[i] = i < nc ? sv.contact[i] : Row{};
    fh[i] = i < nf ? sv.friction[i] : Row{};
  }
  RS_UNROLL
  for (int i = 0; i < HELD_ROWS; ++i)
    if (i < nc) bank.set_applied(i, ch[i].applied);
  for (int i = HELD_ROWS; i < nc; ++i) bank.set_applied(i, sv.contact[i].applied);
  uint32_t run = nc >= 32 ? ~0u : (1u << nc) - 1u;
  for (int it = 0; it < SOLVER_ITERATIONS && run != 0; ++it) {
    RS_UNROLL
    for (int i = 0; i < HELD_ROWS; ++i) {
      if (!((run >> i) & 1u)) continue;
      float res = resolve_split(ch[i], bank);
      if (res * res == 0.0f) run &= ~(1u << i);
    }
    Row next = nc > HELD_ROWS ? sv.contact[HELD_ROWS] : Row{};
    for (int i = HELD_ROWS; i < nc; ++i) {
      Row r = next;
      if (i + 1 < nc) next = sv.contact[i + 1];
      if (!((run >> i) & 1u)) continue;
      float res = resolve_split(r, bank);
      sv.contact[i].applied_push = r.applied_push;
      if (res * res == 0.0f) run &= ~(1u << i);
    }
  }
  for (int it = 0; it < SOLVER_ITERATIONS; ++it) {
    float lsr = 0.0f;
    RS_UNROLL
    for (int i = 0; i < HELD_ROWS; ++i) {
      if (i >= nc || ch[i].split_only) continue;
      float res = resolve_row(ch[i], bank, false);
      bank.set_applied(i, ch[i].applied);
      lsr = fmax_rs(res * res, lsr);
    }
    Row next = nc > HELD_ROWS ? sv.contact[HELD_ROWS] : Row{};
    for (int i = HELD_ROWS; i < nc; ++i) {
      Row r = next;
      if (i + 1 < nc) next = sv.contact[i + 1];
      if (r.split_only) continue;
      float res = resolve_row(r, bank, false);
      sv.contact[i].applied = r.applied;
      bank.set_applied(i, r.applied);
      lsr = fmax_rs(res * res, lsr);
    }
    RS_UNROLL
    for (int i = 0; i < HELD_ROWS; ++i) {
      if (i >= nf) continue;
      float total = bank.applied(fh[i].friction_idx);
      if (total <= 0.0f) continue;
      float lim = fh[i].friction * total;
      fh[i].lower = fneg(lim);
      fh[i].upper = lim;
      float res = resolve_row(fh[i], bank, true);
      lsr = fmax_rs(res * res, lsr);
    }
    next = nf > HELD_ROWS ? sv.friction[HELD_ROWS] : Row{};
    for (int i = HELD_ROWS; i < nf; ++i) {
      Row r = next;
      if (i + 1 < nf) next = sv.friction[i + 1];
      float total = bank.applied(r.friction_idx);
      if (total <= 0.0f) continue;
      float lim = r.friction * total;
      r.lower = fneg(lim);
      r.upper = lim;
      float res = resolve_row(r, bank, true);
      sv.friction[i].lower = r.lower;
      sv.friction[i].upper = r.upper;
      sv.friction[i].applied = r.applied;
      lsr = fmax_rs(res * res, lsr);
    }
    if (lsr == 0.0f) break;
  }
}
RS_FN void solver_finish(const Solver& sv, ArenaState& s, const DeltaBank& bank, float dt) {  // :271-301
  Body b[NUM_DYN];
  RS_UNROLL
  for (int d = 0; d < NUM_DYN; ++d) b[d] = s.bodies[d];
  RS_UNROLL
  for (int d = 0; d < NUM_DYN; ++d) {
    if (!((sv.used >> d) & 1u)) continue;
    Body& body = s.bodies[d];
    const V3 lin = b[d].lin_vel + bank.get(d, BF_DLIN), ang = b[d].ang_vel + bank.get(d, BF_DANG);
    const V3 push = bank.get(d, BF_PUSH), turn = bank.get(d, BF_TURN);
    if (length_sq(push) != 0.0f || length_sq(turn) != 0.0f) {
      Aff t = b[d].world;
      if (b[d].collision_flags & k::CF_NO_ANGULAR_MOTION) {
        t.t += push * dt;
      } else {
        Quat q = b[d].world_quat;
        integrate_trans(&t, &q, push, turn * SPLIT_TURN_ERP, dt);
      }
      set_world_trans(body, t);
    }
    V3 lv = lin + b[d].accum_lin_vel, av = ang + b[d].accum_ang_vel;
    body.lin_vel = lv;
    body.ang_vel = av;
    if (b[d].activation == k::ACT_SLEEPING && (lv.x != 0.0f || lv.y != 0.0f || lv.z != 0.0f || av.x != 0.0f || av.y != 0.0f || av.z != 0.0f)) {
      set_activation(body, k::ACT_WANTS_DEACTIVATION);
      body.deactivation_time = 0.0f;
    }
  }
}
RS_INLINE void phase_p5(ArenaState& s, const StaticData& w) {
  const float dt = 1.0f / 120.0f;
  Solver sv;
  sv.n_contact = sv.n_friction = 0;
  solver_setup(sv, s, w, dt);
  DeltaBank bank;
  solver_iterate(sv, w, bank);
  solver_finish(sv, s, bank, dt);
}

}  // namespace rs
