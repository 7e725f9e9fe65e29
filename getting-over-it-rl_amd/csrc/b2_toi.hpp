// b2_toi.hpp - continuous collision on the device: b2World::SolveTOI with b2TimeOfImpact, b2Distance (GJK),
// b2SeparationFunction, b2Sweep::Advance and b2Island::SolveTOI (goi_jax/box2d/toi.py:73-865). Each world's lane
// group runs its event loop; the sweeps live in the State leaves (c0, c, a0, a, toi.alpha0).
#pragma once

#include "b2_joints.hpp"

namespace goi {

struct Sweep {
    V2 lc, c0, c;
    float a0, a;
};

// b2Sweep::GetTransform (toi.py:73-81); the rotation through the sweep's memo
GOI_D Xf sweep_xf(const Sweep& sw, float beta, RotMemo& memo) {
    Xf t;
    const float omb = 1.0f - beta;
    t.q = memo.of(omb * sw.a0 + beta * sw.a);
    t.p = mk(omb * sw.c0.x + beta * sw.c.x, omb * sw.c0.y + beta * sw.c.y) - mul(t.q, sw.lc);
    return t;
}

GOI_D Sweep body_sweep(const World& W, int b) {
    Sweep s;
    s.lc = W.v2(GOI_B_LOCAL_CENTER, b);
    s.c0 = W.v2(GOI_B_C0, b);
    s.c = W.v2(GOI_B_C, b);
    s.a0 = W.f(GOI_B_A0, b);
    s.a = W.f(GOI_B_A, b);
    return s;
}

// b2Sweep::Advance on body b's sweep (toi.py:100-104)
GOI_D void sweep_advance(const World& W, int b, float alpha) {
    const float al0 = W.f(GOI_T_ALPHA0, b);
    const float den = 1.0f - al0;
    const float beta = (alpha - al0) / (den != 0.0f ? den : 1.0f);
    const V2 c0 = W.v2(GOI_B_C0, b), c = W.v2(GOI_B_C, b);
    W.set2(GOI_B_C0, b, c0 + beta * (c - c0));
    const float a0 = W.f(GOI_B_A0, b);
    W.f(GOI_B_A0, b) = a0 + beta * (W.f(GOI_B_A, b) - a0);
    W.f(GOI_T_ALPHA0, b) = alpha;
}

// b2Body::SynchronizeTransform
GOI_D void sync_transform(const World& W, int b) {
    const float a = W.f(GOI_B_A, b);
    Rot q;
    if (a == 0.0f) {  // a static body's usual angle: rot_of's result, sin = the angle itself (+-0), cos = 1
        q.s = a;
        q.c = 1.0f;
    } else {
        q = rot_of(a);
    }
    W.set2(GOI_B_XF_P, b, W.v2(GOI_B_C, b) - mul(q, W.v2(GOI_B_LOCAL_CENTER, b)));
    W.f(GOI_B_XF_Q, 2 * b) = q.c;
    W.f(GOI_B_XF_Q, 2 * b + 1) = q.s;
}

// b2Body::Advance
GOI_D void body_advance(const World& W, int b, float alpha) {
    sweep_advance(W, b, alpha);
    W.set2(GOI_B_C, b, W.v2(GOI_B_C0, b));
    W.f(GOI_B_A, b) = W.f(GOI_B_A0, b);
    sync_transform(W, b);
}

struct SweepBackup {
    V2 c0, c;
    float a0, a, alpha0;
};
GOI_D SweepBackup backup(const World& W, int b) {
    SweepBackup k;
    k.c0 = W.v2(GOI_B_C0, b); k.c = W.v2(GOI_B_C, b);
    k.a0 = W.f(GOI_B_A0, b); k.a = W.f(GOI_B_A, b); k.alpha0 = W.f(GOI_T_ALPHA0, b);
    return k;
}
GOI_D void restore(const World& W, int b, const SweepBackup& k) {
    W.set2(GOI_B_C0, b, k.c0); W.set2(GOI_B_C, b, k.c);
    W.f(GOI_B_A0, b) = k.a0; W.f(GOI_B_A, b) = k.a; W.f(GOI_T_ALPHA0, b) = k.alpha0;
    sync_transform(W, b);
}

// ---------------------------------------------------------------- distance proxies and GJK (toi.py:116-294)

// b2DistanceProxy held in registers: the fixture's 8 vertex slots are loaded once, in one batch, so GJK's support
// searches stay off memory. The slots past the count repeat vertex 0, which a search for the first largest dot never
// selects over it, so the searches need no test against the count.
struct Proxy {
    V2 v[kPoly];
    int count;
    float radius;
};
GOI_D Proxy proxy_of(const DModel& m, int f) {
    Proxy p;
    p.count = m.fix[f].count;
    p.radius = m.fix[f].radius;
#pragma unroll
    for (int j = 0; j < kPoly; ++j) {
        p.v[j] = m.poly[16 * f + j];
        if (j > 0 && j >= p.count) p.v[j] = p.v[0];
    }
    return p;
}
// b2DistanceProxy::GetSupport and GetVertex together: the first index of the largest dot and its vertex, selected in
// the same pass over the slots (no select chain over the slots by index after it); a quad's pass covers 4 slots
struct Support {
    V2 v;
    int i;
};
template <int kFrom, int kTo>
GOI_D void support_over(const Proxy& p, V2 d, Support& s, float& bv) {
#pragma unroll
    for (int i = kFrom; i < kTo; ++i) {
        const float v = dot(p.v[i], d);
        if (v > bv) {
            s.i = i;
            s.v = p.v[i];
            bv = v;
        }
    }
}
GOI_D Support support(const Proxy& p, V2 d) {
    Support s;
    s.i = 0;
    s.v = p.v[0];
    float bv = dot(p.v[0], d);
    support_over<1, 4>(p, d, s, bv);
    if (p.count > 4) support_over<4, kPoly>(p, d, s, bv);
    return s;
}

// A simplex vertex, with the proxies' own vertices beside their indices, so that neither GJK's next call nor the
// separation function looks them up by index (a chain of 24 selects); the witness points follow from them when GJK ends.
struct SVert {
    V2 w, lA, lB;
    float a;
    int iA, iB;
};
struct SimplexCache {
    float metric;
    int count;
    int iA[3], iB[3];
    V2 lA[3], lB[3];
};

GOI_D float metric(const SVert* v, int count) {
    if (count == 2) return length(v[0].w - v[1].w);
    if (count == 3) return cross(v[1].w - v[0].w, v[2].w - v[0].w);
    return 0.0f;
}

GOI_D void set_vertex(SVert& v, const Xf& xA, int iA, V2 lA, const Xf& xB, int iB, V2 lB) {
    v.iA = iA;
    v.iB = iB;
    v.lA = lA;
    v.lB = lB;
    v.w = mul(xB, lB) - mul(xA, lA);
}
// b2Simplex::Solve2 and Solve3 (count 2 or 3): the region of the origin first, then one division and selects, so that
// lanes in different regions share their instructions (as branches, the regions of a wave's lanes ran one after another).
// The barycentric coordinates of the slots past the new count stay as Box2D leaves them.
GOI_D void simplex_solve(SVert* v, int& count) {
    enum { kV1, kV2, kV3, kE12, kE13, kE23, kFace };
    const V2 w1 = v[0].w, w2 = v[1].w;
    const V2 e12 = w2 - w1;
    const float d12_1 = dot(w2, e12), d12_2 = -dot(w1, e12);
    int region = d12_2 <= 0.0f ? kV1 : d12_1 <= 0.0f ? kV2 : kE12;
    float p = d12_1, q = d12_2, r = 0.0f, den = d12_1 + d12_2;
    if (count == 3) {
        const V2 w3 = v[2].w;
        const V2 e13 = w3 - w1, e23 = w3 - w2;
        const float d13_1 = dot(w3, e13), d13_2 = -dot(w1, e13);
        const float d23_1 = dot(w3, e23), d23_2 = -dot(w2, e23);
        const float n123 = cross(e12, e13);
        const float d123_1 = n123 * cross(w2, w3), d123_2 = n123 * cross(w3, w1), d123_3 = n123 * cross(w1, w2);
        // the first that holds, in Box2D's order
        region = kFace;
        if ((int)(d23_1 > 0.0f) & (int)(d23_2 > 0.0f) & (int)(d123_1 <= 0.0f)) region = kE23;
        if ((int)(d13_1 <= 0.0f) & (int)(d23_1 <= 0.0f)) region = kV3;
        if ((int)(d12_1 <= 0.0f) & (int)(d23_2 <= 0.0f)) region = kV2;
        if ((int)(d13_1 > 0.0f) & (int)(d13_2 > 0.0f) & (int)(d123_2 <= 0.0f)) region = kE13;
        if ((int)(d12_1 > 0.0f) & (int)(d12_2 > 0.0f) & (int)(d123_3 <= 0.0f)) region = kE12;
        if ((int)(d12_2 <= 0.0f) & (int)(d13_2 <= 0.0f)) region = kV1;
        p = region == kE13 ? d13_1 : region == kE23 ? d23_1 : region == kFace ? d123_1 : p;
        q = region == kE13 ? d13_2 : region == kE23 ? d23_2 : region == kFace ? d123_2 : q;
        r = d123_3;
        den = region == kFace ? (p + q) + r : p + q;
    }
    const float inv = 1.0f / den;
    const bool edge = region >= kE12;
    p = edge ? p * inv : 1.0f;
    q = edge ? q * inv : 1.0f;
    // slot 0 takes vertex 2 (kV2) or 3 (kV3, kE23), slot 1 vertex 3 (kE13)
    const float a1 = v[1].a, a2 = v[2].a;
    const bool from2 = region == kV2, from3 = (region == kV3) | (region == kE23), one3 = region == kE13;
    const auto take = [&](SVert& x, const SVert& y) { x.w = y.w; x.lA = y.lA; x.lB = y.lB; x.iA = y.iA; x.iB = y.iB; };
    if (from2) take(v[0], v[1]);
    if (from3) take(v[0], v[2]);
    if (one3) take(v[1], v[2]);
    v[0].a = region == kE23 ? q : p;
    v[1].a = region == kE23 ? p : (region == kV1) | (region == kV3) ? a1 : q;
    v[2].a = region == kFace ? r * inv : (region == kV3) | (region == kE13) | (region == kE23) ? q : a2;
    count = region < kE12 ? 1 : region == kFace ? 3 : 2;
}

// b2Distance (useRadii = false): the distance and the updated simplex cache. The simplex, the saved indices and
// the cache are indexed only by constants once the short loops are unrolled, so they stay in registers (a runtime
// index would put them in private scratch memory, one memory round trip per access).
GOI_D float gjk_distance(SimplexCache& cache, const Proxy& pA, const Xf& xA, const Proxy& pB, const Xf& xB) {
    SVert v[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        v[i].a = 0.0f;
        v[i].iA = 0; v[i].iB = 0;
        v[i].w = v[i].lA = v[i].lB = mk(0.0f, 0.0f);
    }
    int count = cache.count;
#pragma unroll
    for (int i = 0; i < 3; ++i)
        if (i < count) set_vertex(v[i], xA, cache.iA[i], cache.lA[i], xB, cache.iB[i], cache.lB[i]);
    if (count > 1) {
        const float m1 = cache.metric, m2 = metric(v, count);
        if (m2 < 0.5f * m1 || 2.0f * m1 < m2 || m2 < kEps) count = 0;
    }
    if (count == 0) {
        set_vertex(v[0], xA, 0, pA.v[0], xB, 0, pB.v[0]);
        v[0].a = 1.0f;
        count = 1;
    }
    int saveA[3], saveB[3];
    for (int iter = 0; iter < 20;) {
        const int save = count;
#pragma unroll
        for (int i = 0; i < 3; ++i)
            if (i < save) { saveA[i] = v[i].iA; saveB[i] = v[i].iB; }
        if (count > 1) simplex_solve(v, count);
        if (count == 3) break;
        V2 d;
        if (count == 1) {
            d = -v[0].w;
        } else {
            const V2 e12 = v[1].w - v[0].w;
            d = cross(e12, -v[0].w) > 0.0f ? cross(1.0f, e12) : cross(e12, 1.0f);
        }
        if (dot(d, d) < kEps * kEps) break;
        // the new vertex takes slot `count` (1 or 2); its barycentric coordinate is left as it was
        SVert nv;
        const Support sa = support(pA, mulT(xA.q, -d)), sb = support(pB, mulT(xB.q, d));
        set_vertex(nv, xA, sa.i, sa.v, xB, sb.i, sb.v);
        nv.a = count == 1 ? v[1].a : v[2].a;
        if (count == 1) v[1] = nv;
        else v[2] = nv;
        ++iter;
        bool dup = false;
#pragma unroll
        for (int i = 0; i < 3; ++i)
            if (i < save) dup |= (nv.iA == saveA[i] && nv.iB == saveB[i]);
        if (dup) break;
        ++count;
    }
    const V2 a0 = mul(xA, v[0].lA), b0 = mul(xB, v[0].lB);
    V2 pa = a0, pb = b0;
    if (count > 1) {
        const V2 a1 = mul(xA, v[1].lA), b1 = mul(xB, v[1].lB);
        pa = v[0].a * a0 + v[1].a * a1;
        pb = v[0].a * b0 + v[1].a * b1;
    }
    if (count == 3) {
        pa = pa + v[2].a * mul(xA, v[2].lA);
        pb = pa;
    }
    cache.metric = metric(v, count);
    cache.count = count;
#pragma unroll
    for (int i = 0; i < 3; ++i)
        if (i < count) { cache.iA[i] = v[i].iA; cache.iB[i] = v[i].iB; cache.lA[i] = v[i].lA; cache.lB[i] = v[i].lB; }
    return length(pa - pb);
}

// ---------------------------------------------------------------- b2SeparationFunction and b2TimeOfImpact

enum { kSepPoints = 0, kSepFaceA = 1, kSepFaceB = 2 };
struct SepFn {
    int type;
    V2 axis, lp;
};

// The separation function of the simplex GJK ended with; xA, xB: the sweeps' transforms at t1, where it ran. A face of
// A and a face of B take the same instructions with the two sides exchanged (lanes of different types do not diverge).
GOI_D SepFn sep_init(const SimplexCache& cache, const Xf& xA, const Xf& xB) {
    SepFn f;
    const bool points = cache.count == 1;
    const bool faceB = cache.iA[0] == cache.iA[1];
    f.type = points ? kSepPoints : faceB ? kSepFaceB : kSepFaceA;
    const V2 u1 = faceB ? cache.lB[0] : cache.lA[0], u2 = faceB ? cache.lB[1] : cache.lA[1];  // the face
    const V2 a0 = mul(xA, cache.lA[0]), b0 = mul(xB, cache.lB[0]);
    f.axis = points ? b0 - a0 : cross(u2 - u1, 1.0f);
    normalize(f.axis);
    f.lp = mk(0.0f, 0.0f);
    if (!points) {
        const Xf& own = faceB ? xB : xA;
        const V2 n = mul(own.q, f.axis);
        f.lp = 0.5f * (u1 + u2);
        if (dot((faceB ? a0 : b0) - mul(own, f.lp), n) < 0.0f) f.axis = -f.axis;
    }
    return f;
}

// b2SeparationFunction::Evaluate at the local points lA, lB that FindMinSeparation chose: the support vertices, and a
// face's own point on its side
GOI_D float sep_at(const SepFn& f, const Xf& xA, const Xf& xB, V2 n, V2 lA, V2 lB) {
    const V2 pA = mul(xA, lA), pB = mul(xB, lB);
    const bool faceB = f.type == kSepFaceB;
    return dot((faceB ? pA : pB) - (faceB ? pB : pA), n);
}
GOI_D V2 sep_normal(const SepFn& f, const Xf& xA, const Xf& xB) {
    const V2 n = mul(f.type == kSepFaceB ? xB.q : xA.q, f.axis);
    return f.type == kSepPoints ? f.axis : n;
}
GOI_D float sep_eval(const SepFn& f, const Xf& xA, const Xf& xB, V2 lA, V2 lB) {
    return sep_at(f, xA, xB, sep_normal(f, xA, xB), lA, lB);
}

// b2SeparationFunction::FindMinSeparation; lA, lB: its support vertices, the face's point on a face's own side
GOI_D float sep_find_min(const SepFn& f, const Proxy& pA, const Sweep& sA, const Proxy& pB, const Sweep& sB, V2& lA,
                         V2& lB, float t, RotMemo& ma, RotMemo& mb) {
    const Xf xA = sweep_xf(sA, t, ma), xB = sweep_xf(sB, t, mb);
    const V2 n = sep_normal(f, xA, xB);
    lA = support(pA, mulT(xA.q, f.type == kSepPoints ? n : -n)).v;
    lB = support(pB, mulT(xB.q, -n)).v;
    if (f.type == kSepFaceA) lA = f.lp;
    if (f.type == kSepFaceB) lB = f.lp;
    return sep_at(f, xA, xB, n, lA, lB);
}

enum { kToiUnknown = 0, kToiFailed = 1, kToiOverlapped = 2, kToiTouching = 3, kToiSeparated = 4 };

// b2TimeOfImpact with tMax = 1 (toi.py:364-457): separating axes (20), push-backs (8), root finder (50 steps of
// alternating bisection and secant)
GOI_D int time_of_impact(const Proxy& pA, Sweep sA, const Proxy& pB, Sweep sB, float linear_slop, float& t_out) {
    const float two_pi = 2.0f * kPi;
    {
        const float d = two_pi * floorf(sA.a0 / two_pi);
        sA.a0 = sA.a0 - d; sA.a = sA.a - d;
    }
    {
        const float d = two_pi * floorf(sB.a0 / two_pi);
        sB.a0 = sB.a0 - d; sB.a = sB.a - d;
    }
    const float total_radius = pA.radius + pB.radius;
    const float target = bmax(linear_slop, total_radius - 3.0f * linear_slop);
    const float tol = 0.25f * linear_slop;
    float t1 = 0.0f;
    SimplexCache cache;
    cache.count = 0;
    cache.metric = 0.0f;
    int state = kToiUnknown;
    t_out = 1.0f;
    RotMemo ma, mb;
    for (int iter = 0;;) {
        const Xf xA1 = sweep_xf(sA, t1, ma), xB1 = sweep_xf(sB, t1, mb);
        const float dist = gjk_distance(cache, pA, xA1, pB, xB1);
        if (dist <= 0.0f) { state = kToiOverlapped; t_out = 0.0f; break; }
        if (dist < target + tol) { state = kToiTouching; t_out = t1; break; }
        const SepFn f = sep_init(cache, xA1, xB1);
        bool done = false;
        float t2 = 1.0f;
        for (int push = 0;;) {
            V2 lA, lB;
            float s2 = sep_find_min(f, pA, sA, pB, sB, lA, lB, t2, ma, mb);
            if (s2 > target + tol) { state = kToiSeparated; t_out = 1.0f; done = true; break; }
            if (s2 > target - tol) { t1 = t2; break; }
            float s1 = sep_eval(f, xA1, xB1, lA, lB);
            if (s1 < target - tol) { state = kToiFailed; t_out = t1; done = true; break; }
            if (s1 <= target + tol) { state = kToiTouching; t_out = t1; done = true; break; }
            float a1 = t1, a2 = t2;
            for (int rc = 0;;) {
                const float t = (rc & 1) ? a1 + (target - s1) * (a2 - a1) / (s2 - s1) : 0.5f * (a1 + a2);
                ++rc;
                const float s = sep_eval(f, sweep_xf(sA, t, ma), sweep_xf(sB, t, mb), lA, lB);
                if (babs(s - target) < tol) { t2 = t; break; }
                if (s > target) { a1 = t; s1 = s; }
                else { a2 = t; s2 = s; }
                if (rc == 50) break;
            }
            if (++push == kPoly) break;
        }
        ++iter;
        if (done) break;
        if (iter == 20) { state = kToiFailed; t_out = t1; break; }
    }
    return state;
}

}  // namespace goi
