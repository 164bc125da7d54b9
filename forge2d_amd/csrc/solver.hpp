// Restates algorithms of Box2D v3.1.1, MIT License, Copyright (c) 2022 Erin Catto (THIRD_PARTY_NOTICES).
// Contact and body solver stages, one constraint (or body) per lane.
//
// Coloured constraints follow the 4-wide SIMD solver's per-lane arithmetic
// (S/contact_solver.c:1438-2120): b2MulAddW(a,b,c) = a + b*c, b2MulSubW = a - b*c,
// b2MaxW/b2MinW = SSE max/min (a > b ? a : b, a < b ? a : b), blends on the sign
// of s > 0. Overflow constraints follow the scalar solver (:24-509), whose
// expression order differs (impulse formula, minimum bias velocity, clamps).
// Body integration follows S/solver.c:65-198 and finalize :543-726.
#pragma once

#include "layout.hpp"

namespace f2d {

#if defined(__HIP_DEVICE_COMPILE__)
F2D_HD float asFloat(int v) { return __int_as_float(v); }
F2D_HD int asInt(float v) { return __float_as_int(v); }
#else
inline float asFloat(int v) {
  float f;
  __builtin_memcpy(&f, &v, 4);
  return f;
}
inline int asInt(float v) {
  int i;
  __builtin_memcpy(&i, &v, 4);
  return i;
}
#endif

struct Cons {
  float* f;
  long stride;
  F2D_HD float4& group(int g, long lane) const { return reinterpret_cast<float4*>(f)[g * stride + lane]; }
  F2D_HD float& at(int field, long lane) const { return f[4 * ((field >> 2) * stride + lane) + (field & 3)]; }
  F2D_HD int geti(int field, long lane) const { return asInt(at(field, lane)); }
  F2D_HD void seti(int field, long lane, int v) const { at(field, lane) = asFloat(v); }
};

F2D_HD BodyState identityState() {
  BodyState s;
  s.v = {0.0f, 0.0f};
  s.w = 0.0f;
  s.flags = 0;
  s.dp = {0.0f, 0.0f};
  s.dq = {1.0f, 0.0f};
  return s;
}

#if defined(__HIP_DEVICE_COMPILE__)
#define F2D_UNROLL2 _Pragma("unroll")
#else
#define F2D_UNROLL2
#endif

// One contact constraint's terms of the substeps, in registers.
struct ContactLane {
  float nx, ny, friction, tangentSpeed, rollingRes, rollingMass, rollingImpulse;
  float ax[2], ay[2], bx[2], by[2];  // anchors
  float sep[2], nm[2], tm[2];        // base separation, normal and tangent mass
  float ni[2], ti[2], tni[2];        // normal, tangent and total normal impulses
};
// The inverse masses and inertias of its bodies (zero for a static body)
struct ContactMass {
  float mA, iA, mB, iB;
};

// ---------------------------------------------------------------------------- prepare

// b2PrepareContactsTask lane body, S/contact_solver.c:1462-1627 (identical to the
// overflow prepare :50-157 for the quantities both compute). relVel: the points'
// relative normal velocities.
F2D_HD void prepareLane(ContactLane& c, const Contact& cs, const ContactMass& k, const BodyState& sA,
                        const BodyState& sB, float warmStartScale, float* relVel) {
  const Manifold& m = cs.m;
  const float mA = k.mA, iA = k.iA, mB = k.mB, iB = k.iB;
  {
    float i = iA + iB;
    c.rollingMass = i > 0.0f ? 1.0f / i : 0.0f;
  }
  Vec2 normal = m.normal;
  c.nx = normal.x;
  c.ny = normal.y;
  c.friction = cs.friction;
  c.tangentSpeed = cs.tangentSpeed;
  c.rollingRes = cs.rollingResistance;
  c.rollingImpulse = warmStartScale * m.rollingImpulse;
  Vec2 tangent = rightPerp(normal);
  const int pointCount = m.pointCount;
  F2D_UNROLL2
  for (int p = 0; p < 2; ++p) {
    if (p < pointCount) {
      const ManifoldPoint& mp = m.points[p];
      Vec2 rA = mp.anchorA;
      Vec2 rB = mp.anchorB;
      c.ax[p] = rA.x;
      c.ay[p] = rA.y;
      c.bx[p] = rB.x;
      c.by[p] = rB.y;
      c.sep[p] = mp.separation - dot(sub(rB, rA), normal);
      c.ni[p] = warmStartScale * mp.normalImpulse;
      c.ti[p] = warmStartScale * mp.tangentImpulse;
      float rnA = cross(rA, normal);
      float rnB = cross(rB, normal);
      float kNormal = mA + mB + iA * rnA * rnA + iB * rnB * rnB;
      c.nm[p] = kNormal > 0.0f ? 1.0f / kNormal : 0.0f;
      float rtA = cross(rA, tangent);
      float rtB = cross(rB, tangent);
      float kTangent = mA + mB + iA * rtA * rtA + iB * rtB * rtB;
      c.tm[p] = kTangent > 0.0f ? 1.0f / kTangent : 0.0f;
      Vec2 vrA = add(sA.v, crossSV(sA.w, rA));
      Vec2 vrB = add(sB.v, crossSV(sB.w, rB));
      relVel[p] = dot(normal, sub(vrB, vrA));
    } else {
      c.ax[p] = c.ay[p] = c.bx[p] = c.by[p] = 0.0f;
      c.sep[p] = c.nm[p] = c.tm[p] = c.ni[p] = c.ti[p] = 0.0f;
      relVel[p] = 0.0f;
    }
    c.tni[p] = 0.0f;
  }
}

// ---------------------------------------------------------------------------- coloured (SIMD lane order)

// b2WarmStartContactsTask lane, S/contact_solver.c:1671-1727
F2D_HD void warmStartCore(const ContactLane& c, const ContactMass& k, BodyState& bA, BodyState& bB) {
  float tx = c.ny;
  float ty = 0.0f - c.nx;
  F2D_UNROLL2
  for (int p = 0; p < 2; ++p) {
    float Px = c.ni[p] * c.nx + c.ti[p] * tx;
    float Py = c.ni[p] * c.ny + c.ti[p] * ty;
    bA.w = bA.w - k.iA * (c.ax[p] * Py - c.ay[p] * Px);
    bA.v.x = bA.v.x - k.mA * Px;
    bA.v.y = bA.v.y - k.mA * Py;
    bB.w = bB.w + k.iB * (c.bx[p] * Py - c.by[p] * Px);
    bB.v.x = bB.v.x + k.mB * Px;
    bB.v.y = bB.v.y + k.mB * Py;
  }
  bA.w = bA.w - k.iA * c.rollingImpulse;
  bB.w = bB.w + k.iB * c.rollingImpulse;
}

// b2SolveContactsTask lane, S/contact_solver.c:1729-1967; soft: the contact's softness
// (solve) or {0, 1, 0} (relax)
F2D_HD void solveCore(ContactLane& c, const ContactMass& k, BodyState& bA, BodyState& bB, float inv_h,
                      float minBiasVel, Softness soft) {
  const float mA = k.mA, iA = k.iA, mB = k.mB, iB = k.iB;
  const float nx = c.nx, ny = c.ny;
  float totalNormalImpulse = 0.0f;
  float dpx = bB.dp.x - bA.dp.x;
  float dpy = bB.dp.y - bA.dp.y;
  F2D_UNROLL2
  for (int p = 0; p < 2; ++p) {
    float rAx = c.ax[p], rAy = c.ay[p];
    float rBx = c.bx[p], rBy = c.by[p];
    // moving anchors for current separation
    float rsAx = bA.dq.c * rAx - bA.dq.s * rAy;
    float rsAy = bA.dq.s * rAx + bA.dq.c * rAy;
    float rsBx = bB.dq.c * rBx - bB.dq.s * rBy;
    float rsBy = bB.dq.s * rBx + bB.dq.c * rBy;
    float dsx = dpx + (rsBx - rsAx);
    float dsy = dpy + (rsBy - rsAy);
    float s = (nx * dsx + ny * dsy) + c.sep[p];
    bool mask = s > 0.0f;
    float specBias = s * inv_h;
    float softBias = maxf(soft.biasRate * s, minBiasVel);
    float bias = mask ? specBias : softBias;
    float pointMassScale = mask ? 1.0f : soft.massScale;
    float pointImpulseScale = mask ? 0.0f : soft.impulseScale;
    float dvx = (bB.v.x - bB.w * rBy) - (bA.v.x - bA.w * rAy);
    float dvy = (bB.v.y + bB.w * rBx) - (bA.v.y + bA.w * rAx);
    float vn = dvx * nx + dvy * ny;
    float ni = c.ni[p];
    float negImpulse = c.nm[p] * (pointMassScale * (vn + bias)) + pointImpulseScale * ni;
    float newImpulse = maxf(ni - negImpulse, 0.0f);
    float impulse = newImpulse - ni;
    c.ni[p] = newImpulse;
    c.tni[p] = c.tni[p] + newImpulse;
    totalNormalImpulse = totalNormalImpulse + newImpulse;
    float Px = impulse * nx;
    float Py = impulse * ny;
    bA.v.x = bA.v.x - mA * Px;
    bA.v.y = bA.v.y - mA * Py;
    bA.w = bA.w - iA * (rAx * Py - rAy * Px);
    bB.v.x = bB.v.x + mB * Px;
    bB.v.y = bB.v.y + mB * Py;
    bB.w = bB.w + iB * (rBx * Py - rBy * Px);
  }
  float tx = ny;
  float ty = 0.0f - nx;
  F2D_UNROLL2
  for (int p = 0; p < 2; ++p) {
    float rAx = c.ax[p], rAy = c.ay[p];
    float rBx = c.bx[p], rBy = c.by[p];
    float dvx = (bB.v.x - bB.w * rBy) - (bA.v.x - bA.w * rAy);
    float dvy = (bB.v.y + bB.w * rBx) - (bA.v.y + bA.w * rAx);
    float vt = dvx * tx + dvy * ty;
    vt = vt - c.tangentSpeed;
    float negImpulse = c.tm[p] * vt;
    float maxFriction = c.friction * c.ni[p];
    float ti = c.ti[p];
    float newImpulse = ti - negImpulse;
    newImpulse = maxf(0.0f - maxFriction, minf(newImpulse, maxFriction));
    float impulse = newImpulse - ti;
    c.ti[p] = newImpulse;
    float Px = impulse * tx;
    float Py = impulse * ty;
    bA.v.x = bA.v.x - mA * Px;
    bA.v.y = bA.v.y - mA * Py;
    bA.w = bA.w - iA * (rAx * Py - rAy * Px);
    bB.v.x = bB.v.x + mB * Px;
    bB.v.y = bB.v.y + mB * Py;
    bB.w = bB.w + iB * (rBx * Py - rBy * Px);
  }
  {
    float deltaLambda = c.rollingMass * (bA.w - bB.w);
    float lambda = c.rollingImpulse;
    float maxLambda = c.rollingRes * totalNormalImpulse;
    // b2SymClampW: max(-b, min(a, b)) with -b formed by flipping the sign bit
    float a = lambda + deltaLambda;
    float nb = -maxLambda;
    float ri = maxf(nb, minf(a, maxLambda));
    c.rollingImpulse = ri;
    deltaLambda = ri - lambda;
    bA.w = bA.w - iA * deltaLambda;
    bB.w = bB.w + iB * deltaLambda;
  }
}

// b2ApplyRestitutionTask lane, S/contact_solver.c:1969-2076. A lane with zero
// restitution is skipped by the callers: in the 4-wide code such a lane is masked to
// zero mass, which leaves its impulses and velocities unchanged.
F2D_HD void restitutionCore(ContactLane& c, const ContactMass& k, BodyState& bA, BodyState& bB, float restitution,
                            const float* relVel, float threshold) {
  F2D_UNROLL2
  for (int p = 0; p < 2; ++p) {
    bool mask1 = (relVel[p] + threshold) > 0.0f;
    bool mask2 = c.tni[p] == 0.0f;
    bool mask = mask1 || mask2;
    float mass = mask ? 0.0f : c.nm[p];
    float rAx = c.ax[p], rAy = c.ay[p];
    float rBx = c.bx[p], rBy = c.by[p];
    float dvx = (bB.v.x - bB.w * rBy) - (bA.v.x - bA.w * rAy);
    float dvy = (bB.v.y + bB.w * rBx) - (bA.v.y + bA.w * rAx);
    float vn = dvx * c.nx + dvy * c.ny;
    float negImpulse = mass * (vn + restitution * relVel[p]);
    float ni = c.ni[p];
    float newImpulse = maxf(ni - negImpulse, 0.0f);
    float impulse = newImpulse - ni;
    c.ni[p] = newImpulse;
    float Px = impulse * c.nx;
    float Py = impulse * c.ny;
    bA.v.x = bA.v.x - k.mA * Px;
    bA.v.y = bA.v.y - k.mA * Py;
    bA.w = bA.w - k.iA * (rAx * Py - rAy * Px);
    bB.v.x = bB.v.x + k.mB * Px;
    bB.v.y = bB.v.y + k.mB * Py;
    bB.w = bB.w + k.iB * (rBx * Py - rBy * Px);
  }
}

// b2StoreImpulsesTask lane, S/contact_solver.c:2078-2120 (writes both points)
F2D_HD void storeLane(const ContactLane& c, const float* relVel, Contact& cs) {
  Manifold& m = cs.m;
  m.rollingImpulse = c.rollingImpulse;
  F2D_UNROLL2
  for (int p = 0; p < 2; ++p) {
    m.points[p].normalImpulse = c.ni[p];
    m.points[p].tangentImpulse = c.ti[p];
    m.points[p].totalNormalImpulse = c.tni[p];
    m.points[p].normalVelocity = relVel[p];
  }
}

// ---------------------------------------------------------------------------- lanes in memory

// Static bodies have no solver state: they read the identity state and drop the write
// (S/contact_solver.c:175-176; their inverse mass and inertia are zero, so the scalar
// solver's dummy state never changes either).
F2D_HD BodyState loadState(const BodyState* states, int idx) { return idx < 0 ? identityState() : states[idx]; }
F2D_HD void storeVel(BodyState* states, int idx, Vec2 v, float w) {
  if (idx >= 0) {
    states[idx].v = v;
    states[idx].w = w;
  }
}

// Every field that the solve stages read, loaded together (the loads are issued back to
// back, before the first store of the stage)
F2D_HD void loadLane(const Cons& c, long lane, int4& head, ContactLane& l, ContactMass& k) {
  const float4 g0 = c.group(0, lane), g1 = c.group(1, lane), g2 = c.group(2, lane), g3 = c.group(3, lane),
               g4 = c.group(4, lane), g5 = c.group(5, lane), g6 = c.group(6, lane), g7 = c.group(7, lane),
               g8 = c.group(8, lane);
  head = make_int4(asInt(g0.x), asInt(g0.y), asInt(g0.z), asInt(g0.w));
  l.nx = g1.x, l.ny = g1.y, l.friction = g1.z, l.tangentSpeed = g1.w;
  l.ax[0] = g2.x, l.ay[0] = g2.y, l.bx[0] = g2.z, l.by[0] = g2.w;
  l.ax[1] = g3.x, l.ay[1] = g3.y, l.bx[1] = g3.z, l.by[1] = g3.w;
  l.sep[0] = g4.x, l.sep[1] = g4.y, l.nm[0] = g4.z, l.nm[1] = g4.w;
  l.tm[0] = g5.x, l.tm[1] = g5.y, l.rollingRes = g5.z, l.rollingMass = g5.w;
  l.ni[0] = g6.x, l.ti[0] = g6.y, l.ni[1] = g6.z, l.ti[1] = g6.w;
  l.tni[0] = g7.x, l.tni[1] = g7.y, l.rollingImpulse = g7.z;
  k.mA = g8.x, k.iA = g8.y, k.mB = g8.z, k.iB = g8.w;
}
F2D_HD void storeLaneImpulses(const Cons& c, long lane, const ContactLane& l) {
  c.group(6, lane) = make_float4(l.ni[0], l.ti[0], l.ni[1], l.ti[1]);
  c.group(7, lane) = make_float4(l.tni[0], l.tni[1], l.rollingImpulse, 0.0f);
}

// indexA, indexB: solver state of each body, -1 for a static one
F2D_HD void prepareMemoryLane(const Cons& c, long lane, const Contact& cs, int slot, int indexA, int indexB,
                              const ContactMass& k, const BodyState* states, float warmStartScale) {
  ContactLane l;
  float relVel[2];
  prepareLane(l, cs, k, loadState(states, indexA), loadState(states, indexB), warmStartScale, relVel);
  c.group(0, lane) = make_float4(asFloat(indexA), asFloat(indexB), asFloat(slot), asFloat(cs.m.pointCount));
  c.group(1, lane) = make_float4(l.nx, l.ny, l.friction, l.tangentSpeed);
  c.group(2, lane) = make_float4(l.ax[0], l.ay[0], l.bx[0], l.by[0]);
  c.group(3, lane) = make_float4(l.ax[1], l.ay[1], l.bx[1], l.by[1]);
  c.group(4, lane) = make_float4(l.sep[0], l.sep[1], l.nm[0], l.nm[1]);
  c.group(5, lane) = make_float4(l.tm[0], l.tm[1], l.rollingRes, l.rollingMass);
  storeLaneImpulses(c, lane, l);
  c.group(8, lane) = make_float4(k.mA, k.iA, k.mB, k.iB);
  c.group(9, lane) = make_float4(cs.restitution, relVel[0], relVel[1], 0.0f);
}

F2D_HD void warmStartMemoryLane(const Cons& c, long lane, BodyState* states) {
  int4 head;
  ContactLane l;
  ContactMass k;
  loadLane(c, lane, head, l, k);
  BodyState bA = loadState(states, head.x), bB = loadState(states, head.y);
  warmStartCore(l, k, bA, bB);
  storeVel(states, head.x, bA.v, bA.w);
  storeVel(states, head.y, bB.v, bB.w);
}

// contactSoft, staticSoft: the softness between two bodies and against a static one
F2D_HD void solveMemoryLane(const Cons& c, long lane, BodyState* states, float inv_h, float minBiasVel, bool useBias,
                            Softness contactSoft, Softness staticSoft) {
  int4 head;
  ContactLane l;
  ContactMass k;
  loadLane(c, lane, head, l, k);
  BodyState bA = loadState(states, head.x), bB = loadState(states, head.y);
  const Softness relax = {0.0f, 1.0f, 0.0f};
  solveCore(l, k, bA, bB, inv_h, minBiasVel, useBias ? ((head.x < 0 || head.y < 0) ? staticSoft : contactSoft) : relax);
  storeLaneImpulses(c, lane, l);
  storeVel(states, head.x, bA.v, bA.w);
  storeVel(states, head.y, bB.v, bB.w);
}

F2D_HD void restitutionMemoryLane(const Cons& c, long lane, BodyState* states, float threshold) {
  const float4 g9 = c.group(9, lane);
  if (g9.x == 0.0f) return;
  const float relVel[2] = {g9.y, g9.z};
  int4 head;
  ContactLane l;
  ContactMass k;
  loadLane(c, lane, head, l, k);
  BodyState bA = loadState(states, head.x), bB = loadState(states, head.y);
  restitutionCore(l, k, bA, bB, g9.x, relVel, threshold);
  storeLaneImpulses(c, lane, l);
  storeVel(states, head.x, bA.v, bA.w);
  storeVel(states, head.y, bB.v, bB.w);
}

F2D_HD void storeMemoryLane(const Cons& c, long lane, Contact& cs) {
  int4 head;
  ContactLane l;
  ContactMass k;
  loadLane(c, lane, head, l, k);
  const float4 g9 = c.group(9, lane);
  const float relVel[2] = {g9.y, g9.z};
  storeLane(l, relVel, cs);
}

// ---------------------------------------------------------------------------- overflow (scalar order)

// b2WarmStartOverflowContacts body, S/contact_solver.c:160-225
F2D_HD void overflowWarmStart(const Cons& c, long lane, BodyState* states) {
  int4 head;
  ContactLane l;
  ContactMass k;
  loadLane(c, lane, head, l, k);
  const int ia = head.x, ib = head.y, pointCount = head.w;
  BodyState sA = loadState(states, ia);
  BodyState sB = loadState(states, ib);
  Vec2 vA = sA.v;
  float wA = sA.w;
  Vec2 vB = sB.v;
  float wB = sB.w;
  Vec2 normal = {l.nx, l.ny};
  Vec2 tangent = rightPerp(normal);
  F2D_UNROLL2
  for (int p = 0; p < 2; ++p) {
    if (p >= pointCount) break;
    Vec2 rA = {l.ax[p], l.ay[p]};
    Vec2 rB = {l.bx[p], l.by[p]};
    Vec2 P = add(mulSV(l.ni[p], normal), mulSV(l.ti[p], tangent));
    wA -= k.iA * cross(rA, P);
    vA = mulAdd(vA, -k.mA, P);
    wB += k.iB * cross(rB, P);
    vB = mulAdd(vB, k.mB, P);
  }
  wA -= k.iA * l.rollingImpulse;
  wB += k.iB * l.rollingImpulse;
  storeVel(states, ia, vA, wA);
  storeVel(states, ib, vB, wB);
}

// b2SolveOverflowContacts body, S/contact_solver.c:227-380
F2D_HD void overflowSolve(const Cons& c, long lane, BodyState* states, float inv_h, float pushout, bool useBias,
                          Softness contactSoft, Softness staticSoft) {
  int4 head;
  ContactLane l;
  ContactMass k;
  loadLane(c, lane, head, l, k);
  const int ia = head.x, ib = head.y, pointCount = head.w;
  const float mA = k.mA, iA = k.iA, mB = k.mB, iB = k.iB;
  BodyState sA = loadState(states, ia);
  Vec2 vA = sA.v;
  float wA = sA.w;
  Rot dqA = sA.dq;
  BodyState sB = loadState(states, ib);
  Vec2 vB = sB.v;
  float wB = sB.w;
  Rot dqB = sB.dq;
  Vec2 dp = sub(sB.dp, sA.dp);
  Vec2 normal = {l.nx, l.ny};
  Vec2 tangent = rightPerp(normal);
  Softness softness = (ia < 0 || ib < 0) ? staticSoft : contactSoft;
  float totalNormalImpulse = 0.0f;
  F2D_UNROLL2
  for (int p = 0; p < 2; ++p) {
    if (p >= pointCount) break;
    Vec2 rA = {l.ax[p], l.ay[p]};
    Vec2 rB = {l.bx[p], l.by[p]};
    Vec2 ds = add(dp, sub(rotate(dqB, rB), rotate(dqA, rA)));
    float s = l.sep[p] + dot(ds, normal);
    float velocityBias = 0.0f;
    float massScale = 1.0f;
    float impulseScale = 0.0f;
    if (s > 0.0f) {
      velocityBias = s * inv_h;
    } else if (useBias) {
      velocityBias = maxf(softness.biasRate * s, -pushout);
      massScale = softness.massScale;
      impulseScale = softness.impulseScale;
    }
    Vec2 vrA = add(vA, crossSV(wA, rA));
    Vec2 vrB = add(vB, crossSV(wB, rB));
    float vn = dot(sub(vrB, vrA), normal);
    float ni = l.ni[p];
    float impulse = -l.nm[p] * massScale * (vn + velocityBias) - impulseScale * ni;
    float newImpulse = maxf(ni + impulse, 0.0f);
    impulse = newImpulse - ni;
    l.ni[p] = newImpulse;
    l.tni[p] = l.tni[p] + newImpulse;
    totalNormalImpulse += newImpulse;
    Vec2 P = mulSV(impulse, normal);
    vA = mulSub(vA, mA, P);
    wA -= iA * cross(rA, P);
    vB = mulAdd(vB, mB, P);
    wB += iB * cross(rB, P);
  }
  F2D_UNROLL2
  for (int p = 0; p < 2; ++p) {
    if (p >= pointCount) break;
    Vec2 rA = {l.ax[p], l.ay[p]};
    Vec2 rB = {l.bx[p], l.by[p]};
    Vec2 vrB = add(vB, crossSV(wB, rB));
    Vec2 vrA = add(vA, crossSV(wA, rA));
    float vt = dot(sub(vrB, vrA), tangent) - l.tangentSpeed;
    float impulse = l.tm[p] * (-vt);
    float maxFriction = l.friction * l.ni[p];
    float ti = l.ti[p];
    float newImpulse = clampf(ti + impulse, -maxFriction, maxFriction);
    impulse = newImpulse - ti;
    l.ti[p] = newImpulse;
    Vec2 P = mulSV(impulse, tangent);
    vA = mulSub(vA, mA, P);
    wA -= iA * cross(rA, P);
    vB = mulAdd(vB, mB, P);
    wB += iB * cross(rB, P);
  }
  {
    float deltaLambda = -l.rollingMass * (wB - wA);
    float lambda = l.rollingImpulse;
    float maxLambda = l.rollingRes * totalNormalImpulse;
    float ri = clampf(lambda + deltaLambda, -maxLambda, maxLambda);
    l.rollingImpulse = ri;
    deltaLambda = ri - lambda;
    wA -= iA * deltaLambda;
    wB += iB * deltaLambda;
  }
  storeLaneImpulses(c, lane, l);
  storeVel(states, ia, vA, wA);
  storeVel(states, ib, vB, wB);
}

// b2ApplyOverflowRestitution body, S/contact_solver.c:382-478
F2D_HD void overflowRestitution(const Cons& c, long lane, BodyState* states, float threshold) {
  const float4 g9 = c.group(9, lane);
  const float restitution = g9.x;
  if (restitution == 0.0f) return;
  int4 head;
  ContactLane l;
  ContactMass k;
  loadLane(c, lane, head, l, k);
  const int ia = head.x, ib = head.y, pointCount = head.w;
  BodyState sA = loadState(states, ia);
  Vec2 vA = sA.v;
  float wA = sA.w;
  BodyState sB = loadState(states, ib);
  Vec2 vB = sB.v;
  float wB = sB.w;
  Vec2 normal = {l.nx, l.ny};
  F2D_UNROLL2
  for (int p = 0; p < 2; ++p) {
    if (p >= pointCount) break;
    float relVel = p == 0 ? g9.y : g9.z;
    if (relVel > -threshold || l.tni[p] == 0.0f) continue;
    Vec2 rA = {l.ax[p], l.ay[p]};
    Vec2 rB = {l.bx[p], l.by[p]};
    Vec2 vrB = add(vB, crossSV(wB, rB));
    Vec2 vrA = add(vA, crossSV(wA, rA));
    float vn = dot(sub(vrB, vrA), normal);
    float impulse = -l.nm[p] * (vn + restitution * relVel);
    float ni = l.ni[p];
    float newImpulse = maxf(ni + impulse, 0.0f);
    impulse = newImpulse - ni;
    l.ni[p] = newImpulse;
    l.tni[p] = l.tni[p] + impulse;
    Vec2 P = mulSV(impulse, normal);
    vA = mulSub(vA, k.mA, P);
    wA -= k.iA * cross(rA, P);
    vB = mulAdd(vB, k.mB, P);
    wB += k.iB * cross(rB, P);
  }
  storeLaneImpulses(c, lane, l);
  storeVel(states, ia, vA, wA);
  storeVel(states, ib, vB, wB);
}

// b2StoreOverflowImpulses body, S/contact_solver.c:480-509 (writes pointCount points)
F2D_HD void overflowStore(const Cons& c, long lane, Contact& cs) {
  Manifold& m = cs.m;
  int4 head;
  ContactLane l;
  ContactMass k;
  loadLane(c, lane, head, l, k);
  const float4 g9 = c.group(9, lane);
  F2D_UNROLL2
  for (int p = 0; p < 2; ++p) {
    if (p >= m.pointCount) break;
    m.points[p].normalImpulse = l.ni[p];
    m.points[p].tangentImpulse = l.ti[p];
    m.points[p].totalNormalImpulse = l.tni[p];
    m.points[p].normalVelocity = p == 0 ? g9.y : g9.z;
  }
  m.rollingImpulse = l.rollingImpulse;
}

// ---------------------------------------------------------------------------- bodies

// b2IntegrateVelocitiesTask body, S/solver.c:65-129
F2D_HD void integrateVelocity(BodySim& sim, BodyState& state, Vec2 gravity, float h, float maxLinearSpeed,
                              float maxAngularSpeed) {
  float maxLinearSpeedSquared = maxLinearSpeed * maxLinearSpeed;
  float maxAngularSpeedSquared = maxAngularSpeed * maxAngularSpeed;
  Vec2 v = state.v;
  float w = state.w;
  float linearDamping = 1.0f / (1.0f + h * sim.linearDamping);
  float angularDamping = 1.0f / (1.0f + h * sim.angularDamping);
  float gravityScale = sim.invMass > 0.0f ? sim.gravityScale : 0.0f;
  Vec2 linearVelocityDelta = add(mulSV(h * sim.invMass, sim.force), mulSV(h * gravityScale, gravity));
  float angularVelocityDelta = h * sim.invI * sim.torque;
  v = mulAdd(linearVelocityDelta, linearDamping, v);
  w = angularVelocityDelta + angularDamping * w;
  if (dot(v, v) > maxLinearSpeedSquared) {
    float ratio = maxLinearSpeed / length(v);
    v = mulSV(ratio, v);
    sim.flags |= BF_CAPPED_STEP;
  }
  if (w * w > maxAngularSpeedSquared && (sim.flags & BF_ALLOW_FAST_ROTATION) == 0) {
    float ratio = maxAngularSpeed / absf(w);
    w *= ratio;
    sim.flags |= BF_CAPPED_STEP;
  }
  state.v = v;
  state.w = w;
}

// The per-step body terms of b2IntegrateVelocitiesTask (S/solver.c:65-129): the
// terms that do not change across substeps, evaluated once per step with the
// reference's own expressions, so each substep's update is bit-identical to
// recomputing them.
enum : int { BC_STATIC = 1, BC_FAST_ROTATION = 2, BC_CAPPED = 4 };
struct alignas(16) BodyConst {
  Vec2 dv;        // h*invMass*force + h*gravityScale*gravity
  float dw;       // h*invI*torque
  float linDamp;  // 1 / (1 + h*linearDamping)
  float invMass, invI;  // one 8-byte access
  float angDamp;  // 1 / (1 + h*angularDamping)
  int flags;      // BC_*
};

F2D_HD BodyConst makeBodyConst(const BodySim& sim, Vec2 gravity, float h) {
  BodyConst k;
  k.linDamp = 1.0f / (1.0f + h * sim.linearDamping);
  k.angDamp = 1.0f / (1.0f + h * sim.angularDamping);
  float gravityScale = sim.invMass > 0.0f ? sim.gravityScale : 0.0f;
  k.dv = add(mulSV(h * sim.invMass, sim.force), mulSV(h * gravityScale, gravity));
  k.dw = h * sim.invI * sim.torque;
  k.invMass = sim.invMass;
  k.invI = sim.invI;
  // bodies outside the awake set (static or sleeping) take no solver updates
  k.flags = (sim.setIndex != kAwakeSet ? BC_STATIC : 0) | ((sim.flags & BF_ALLOW_FAST_ROTATION) ? BC_FAST_ROTATION : 0);
  return k;
}

// b2IntegrateVelocitiesTask body from the per-step terms
F2D_HD void integrateVelocityConst(BodyConst& k, BodyState& state, float maxLinearSpeed, float maxAngularSpeed) {
  float maxLinearSpeedSquared = maxLinearSpeed * maxLinearSpeed;
  float maxAngularSpeedSquared = maxAngularSpeed * maxAngularSpeed;
  Vec2 v = mulAdd(k.dv, k.linDamp, state.v);
  float w = k.dw + k.angDamp * state.w;
  if (dot(v, v) > maxLinearSpeedSquared) {
    float ratio = maxLinearSpeed / length(v);
    v = mulSV(ratio, v);
    k.flags |= BC_CAPPED;
  }
  if (w * w > maxAngularSpeedSquared && (k.flags & BC_FAST_ROTATION) == 0) {
    float ratio = maxAngularSpeed / absf(w);
    w *= ratio;
    k.flags |= BC_CAPPED;
  }
  state.v = v;
  state.w = w;
}

// b2IntegratePositionsTask body, S/solver.c:182-198
F2D_HD void integratePosition(BodyState& state, float h) {
  state.dq = integrateRotation(state.dq, h * state.w);
  state.dp = mulAdd(state.dp, h, state.v);
}

}  // namespace f2d
