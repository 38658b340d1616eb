// Contacts of one body against a static triangle mesh: a wave per body, a lane
// where a wave can't hold it.
//
// A restatement of the reference's PCM mesh contact generation
// (geomutils/src/pcm/GuPCMContactSphereMesh.cpp:160-501,
// GuPCMTriangleContactGen.cpp, GuPCMContactConvexCommon.h:131-230,
// GuPersistentContactManifold.cpp:1315-1420, 1678-2160) in the shape this
// build gives it:
//  * candidates: the triangles whose bounds meet the body's bounds inflated
//    by the contact distance, found through the mesh's bounding-volume tree
//    and taken in triangle order (at most MESH_MAX_TRIS);
//  * a triangle whose plane has the body's centre behind it is culled (the
//    mesh is one-sided);
//  * a sphere takes the closest point of each triangle: face contacts at
//    once, edge and vertex contacts deferred and taken by distance unless a
//    face or a closer contact already holds that edge or vertex (the
//    reference's edge and vertex caches);
//  * a capsule takes the part of its segment over the triangle (its prism),
//    else the closest boundary point, deferred like a sphere's;
//  * a box or hull takes its face most opposed to the triangle normal,
//    clipped to the triangle's prism, and its deepest vertex when over it;
//  * contacts group into patches by normal (within 0.996, the reference's
//    acceptance); a patch holds MESH_PC contacts before it is reduced to 4
//    (the deepest, the farthest from it, then the extremes across their line);
//    the deepest MESH_MAXP patches become one constraint each (a sphere keeps
//    one contact per patch).
// The C oracle (oracle/pxo.c, tm_*) is the same algorithm in the same
// arithmetic order.
#pragma once
#include "pxh_convex.h"
#include "pxh_kernels.h"

namespace pxh {

constexpr int MESH_PC = 8;
constexpr int MESH_NPATCH = 6;

struct MC { f3 p; float s; };
struct MPatch { f3 n; int count; float maxPen; MC c[MESH_PC + 1]; };
struct MPatches { MPatch p[MESH_NPATCH]; int np; };

PXH_D int meshReduce4(MC* c, int n, f3 nrm)
{
	if (n <= 4)
		return n;
	bool used[MESH_PC + 1];
	for (int i = 0; i < n; i++)
		used[i] = false;
	int i0 = 0;
	for (int i = 1; i < n; i++)
		if (c[i0].s > c[i].s)
			i0 = i;
	used[i0] = true;
	int i1 = -1;
	float best = -1.0f;
	for (int i = 0; i < n; i++)
	{
		if (used[i]) continue;
		const f3 d = c[i].p - c[i0].p;
		const float dd = dot(d, d);
		if (dd > best) { best = dd; i1 = i; }
	}
	used[i1] = true;
	const f3 ax = cross(c[i1].p - c[i0].p, nrm);
	int i2 = -1, i3 = -1;
	float mx = -3.402823466e+38f, mn = 3.402823466e+38f;
	for (int i = 0; i < n; i++)
	{
		if (used[i]) continue;
		const float d = dot(c[i].p - c[i0].p, ax);
		if (d > mx) { mx = d; i2 = i; }
		if (mn > d) { mn = d; i3 = i; }
	}
	used[i2] = true;
	if (i3 == i2 || mx * mn > 0.0f)
	{
		mx = -3.402823466e+38f;
		i3 = -1;
		for (int i = 0; i < n; i++)
		{
			if (used[i]) continue;
			const float d = dot(c[i].p - c[i0].p, ax);
			if (d > mx) { mx = d; i3 = i; }
		}
	}
	const MC a = c[i0], b = c[i1], e = c[i2], f = c[i3];
	c[0] = a; c[1] = b; c[2] = e; c[3] = f;
	return 4;
}

PXH_D void meshAdd(MPatches& P, f3 n, f3 p, float s)
{
	for (int k = 0; k < P.np; k++)
	{
		MPatch& q = P.p[k];
		if (!(dot(q.n, n) > 0.996f))
			continue;
		for (int j = 0; j < q.count; j++)
		{
			const f3 d = q.c[j].p - p;
			if (1e-10f > dot(d, d))
			{
				if (q.c[j].s > s)
				{
					q.c[j].p = p;
					q.c[j].s = s;
				}
				if (q.maxPen > s)
					q.maxPen = s;
				return;
			}
		}
		q.c[q.count].p = p;
		q.c[q.count].s = s;
		q.count++;
		if (q.maxPen > s)
			q.maxPen = s;
		if (q.count > MESH_PC)
			q.count = meshReduce4(q.c, q.count, q.n);
		return;
	}
	int k = P.np;
	if (k == MESH_NPATCH)
	{
		k = 0;
		for (int j = 1; j < MESH_NPATCH; j++)
			if (P.p[j].maxPen > P.p[k].maxPen)
				k = j;
		if (!(P.p[k].maxPen > s))
			return;
	}
	else
		P.np++;
	P.p[k].n = n;
	P.p[k].count = 1;
	P.p[k].maxPen = s;
	P.p[k].c[0].p = p;
	P.p[k].c[0].s = s;
}

// pcmDistancePointTriangleSquared (GuPCMContactSphereMesh.cpp:160-288)
enum { TF_FACE = 0, TF_V0 = 1, TF_V1 = 2, TF_V2 = 3, TF_E01 = 4, TF_E12 = 5, TF_E20 = 6 };
PXH_D float meshPointTri(f3 p, f3 a, f3 b, f3 c, f3& cp, int& fc)
{
	const f3 ab = b - a, ac = c - a, bc = c - b;
	const f3 ap = p - a, bp = p - b, cq = p - c;
	const float d1 = dot(ab, ap), d2 = dot(ac, ap), d3 = dot(ab, bp), d4 = dot(ac, bp), d5 = dot(ab, cq),
	            d6 = dot(ac, cq);
	const float unom = d4 - d3, udenom = d5 - d6;
	const f3 n = cross(ab, ac);
	if (0.0f > d1 && 0.0f > d2) { fc = TF_V0; cp = a; return dot(ap, ap); }
	if (d3 >= 0.0f && d3 >= d4) { fc = TF_V1; cp = b; return dot(bp, bp); }
	if (d6 >= 0.0f && d6 >= d5) { fc = TF_V2; cp = c; return dot(cq, cq); }
	const float vc = dot(n, cross(ap, bp));
	if (0.0f > vc && d1 >= 0.0f && 0.0f > d3)
	{
		fc = TF_E01;
		const f3 q = ab * (d1 / (d1 - d3)) + a;
		cp = q;
		const f3 vv = p - q;
		return dot(vv, vv);
	}
	const float va = dot(n, cross(bp, cq));
	if (0.0f > va && d4 >= d3 && d5 >= d6)
	{
		fc = TF_E12;
		const f3 q = bc * (unom / (unom + udenom)) + b;
		cp = q;
		const f3 vv = p - q;
		return dot(vv, vv);
	}
	const float vb = dot(n, cross(cq, ap));
	if (0.0f > vb && d2 >= 0.0f && 0.0f > d6)
	{
		fc = TF_E20;
		const f3 q = ac * (d2 / (d2 - d6)) + a;
		cp = q;
		const f3 vv = p - q;
		return dot(vv, vv);
	}
	fc = TF_FACE;
	const float t = dot(n, a - p) / dot(n, n);
	const f3 vv = n * t;
	cp = p + vv;
	return dot(vv, vv);
}

// edge and vertex caches (CachedEdge / CachedVertex,
// geomutils/src/mesh/GuTriangleCache.h:38-90): add returns true when new
struct MeshCache
{
	uint64_t e[3 * MESH_MAX_TRIS];
	int v[3 * MESH_MAX_TRIS];
	int ne, nv;
	PXH_D bool edge(int a, int b)
	{
		const uint64_t k = (uint64_t(uint32_t(a < b ? a : b)) << 32) | uint32_t(a < b ? b : a);
		for (int i = 0; i < ne; i++)
			if (e[i] == k) return false;
		e[ne++] = k;
		return true;
	}
	PXH_D bool vertex(int a)
	{
		for (int i = 0; i < nv; i++)
			if (v[i] == a) return false;
		v[nv++] = a;
		return true;
	}
};

struct MeshTri
{
	f3 v[3], n;
	int vi[3];
};

PXH_D MeshTri meshTri(const MeshSet& M, int t)
{
	MeshTri r;
	const float4 a = M.v0[t], b = M.v1[t], c = M.v2[t];
	r.v[0] = mk(a); r.v[1] = mk(b); r.v[2] = mk(c);
	r.vi[0] = __float_as_int(a.w); r.vi[1] = __float_as_int(b.w); r.vi[2] = __float_as_int(c.w);
	r.n = mk(M.n[t]);
	return r;
}

PXH_D void meshCacheTri(MeshCache& C, const MeshTri& t)
{
	C.edge(t.vi[0], t.vi[1]);
	C.edge(t.vi[1], t.vi[2]);
	C.edge(t.vi[2], t.vi[0]);
	C.vertex(t.vi[0]);
	C.vertex(t.vi[1]);
	C.vertex(t.vi[2]);
}

PXH_D bool meshCulled(const MeshTri& t, f3 c) { return 0.0f > dot(c, t.n) - dot(t.v[0], t.n); }

struct MeshDef { f3 p, n; float sq; int fc, t; };

// deferred edge and vertex contacts by distance, each unless its feature is
// held (PCMSphereVsMeshContactGeneration::generateLastContacts); reported on
// the sphere or capsule: p - n r
PXH_D void meshFlushDeferred(const MeshSet& M, MeshDef* d, int nd, MeshCache& C, float r, MPatches& P)
{
	for (int i = 1; i < nd; i++)
	{
		const MeshDef x = d[i];
		int j = i - 1;
		while (j >= 0 && d[j].sq > x.sq)
		{
			d[j + 1] = d[j];
			j--;
		}
		d[j + 1] = x;
	}
	for (int i = 0; i < nd; i++)
	{
		const MeshTri t = meshTri(M, d[i].t);
		const bool e01 = C.edge(t.vi[0], t.vi[1]);
		const bool e12 = C.edge(t.vi[1], t.vi[2]);
		const bool e20 = C.edge(t.vi[2], t.vi[0]);
		const bool v0 = C.vertex(t.vi[0]);
		const bool v1 = C.vertex(t.vi[1]);
		const bool v2 = C.vertex(t.vi[2]);
		const int fc = d[i].fc;
		const bool need = fc == TF_V0 ? v0 : fc == TF_V1 ? v1 : fc == TF_V2 ? v2 : fc == TF_E01 ? e01 : fc == TF_E12 ? e12 : e20;
		if (need)
		{
			const float dist = sqrtf(d[i].sq);
			meshAdd(P, d[i].n, d[i].p - d[i].n * r, dist - r);
		}
	}
}

PXH_D void meshSphere(const MeshSet& M, const int* idx, int nc, f3 c, float r, float cd, MeshCache& C, MeshDef* def,
                      MPatches& P)
{
	const float infl = r + cd;
	const float inflSq = infl * infl;
	C.ne = C.nv = 0;
	int nd = 0;
	for (int k = 0; k < nc; k++)
	{
		const MeshTri t = meshTri(M, idx[k]);
		if (meshCulled(t, c))
			continue;
		f3 cp;
		int fc;
		const float sq = meshPointTri(c, t.v[0], t.v[1], t.v[2], cp, fc);
		if (!(inflSq > sq))
			continue;
		if (fc == TF_FACE)
		{
			meshCacheTri(C, t);
			const float dist = sqrtf(sq);
			meshAdd(P, t.n, c - t.n * r, dist - r);
		}
		else
		{
			def[nd].p = c;
			def[nd].n = normalize(c - cp);
			def[nd].sq = sq;
			def[nd].fc = fc;
			def[nd].t = idx[k];
			nd++;
		}
	}
	meshFlushDeferred(M, def, nd, C, r, P);
}

// inward normals of the triangle's edge planes
PXH_D void meshPrism(const MeshTri& t, f3* m)
{
	for (int k = 0; k < 3; k++)
		m[k] = cross(t.n, t.v[(k + 1) % 3] - t.v[k]);
}

// closest points of segments p1q1, p2q2 (Ericson, Real-Time Collision
// Detection, 5.1.9), as the oracle's seg_closest2
PXH_D float meshSegClosest(f3 p1, f3 q1, f3 p2, f3 q2, f3& c1, f3& c2)
{
	const f3 d1 = q1 - p1, d2 = q2 - p2, r = p1 - p2;
	const float a = dot(d1, d1), e = dot(d2, d2), f = dot(d2, r);
	float s, t;
	if (a <= 1e-20f && e <= 1e-20f) { s = t = 0.0f; }
	else if (a <= 1e-20f) { s = 0.0f; t = fminf(fmaxf(f / e, 0.0f), 1.0f); }
	else
	{
		const float c = dot(d1, r);
		if (e <= 1e-20f) { t = 0.0f; s = fminf(fmaxf(-c / a, 0.0f), 1.0f); }
		else
		{
			const float b = dot(d1, d2), den = a * e - b * b;
			s = den != 0.0f ? fminf(fmaxf((b * f - c * e) / den, 0.0f), 1.0f) : 0.0f;
			t = (b * s + f) / e;
			if (t < 0.0f) { t = 0.0f; s = fminf(fmaxf(-c / a, 0.0f), 1.0f); }
			else if (t > 1.0f) { t = 1.0f; s = fminf(fmaxf((b - c) / a, 0.0f), 1.0f); }
		}
	}
	c1 = p1 + d1 * s;
	c2 = p2 + d2 * t;
	const f3 w = c1 - c2;
	return dot(w, w);
}

PXH_D void meshCapsule(const MeshSet& M, const int* idx, int nc, f3 p0, f3 p1, f3 c, float r, float cd, MeshCache& C,
                       MeshDef* def, MPatches& P)
{
	const float infl = r + cd;
	C.ne = C.nv = 0;
	int nd = 0;
	for (int k = 0; k < nc; k++)
	{
		const MeshTri t = meshTri(M, idx[k]);
		if (meshCulled(t, c))
			continue;
		f3 m[3];
		meshPrism(t, m);
		float t0 = 0.0f, t1 = 1.0f;
		bool empty = false;
		for (int e = 0; e < 3 && !empty; e++)
		{
			const float a = dot(m[e], p0 - t.v[e]), b = dot(m[e], p1 - t.v[e]);
			if (0.0f > a && 0.0f > b)
				empty = true;
			else if (0.0f > a)
			{
				const float u = a / (a - b);
				if (u > t0) t0 = u;
			}
			else if (0.0f > b)
			{
				const float u = a / (a - b);
				if (t1 > u) t1 = u;
			}
		}
		if (!empty && t1 >= t0)
		{
			const f3 d = p1 - p0;
			f3 q[2];
			q[0] = p0 + d * t0;
			q[1] = p0 + d * t1;
			const int nq = t1 > t0 ? 2 : 1;
			bool any = false;
			for (int j = 0; j < nq; j++)
			{
				const float s = dot(q[j] - t.v[0], t.n);
				if (infl > s)
				{
					meshAdd(P, t.n, q[j] - t.n * r, s - r);
					any = true;
				}
			}
			if (any)
				meshCacheTri(C, t);
			continue;
		}
		float best = 3.402823466e+38f;
		f3 bs = p0, bt = p0;
		int bf = TF_E01;
		for (int e = 0; e < 3; e++)
		{
			f3 cs, ct;
			const float sq = meshSegClosest(p0, p1, t.v[e], t.v[(e + 1) % 3], cs, ct);
			if (best > sq)
			{
				best = sq;
				bs = cs;
				bt = ct;
				bf = e == 0 ? TF_E01 : e == 1 ? TF_E12 : TF_E20;
			}
		}
		if (!(infl * infl > best) || !(best > 0.0f))
			continue;
		const f3 nn = normalize(bs - bt);
		if (!(dot(nn, t.n) > 0.0f))
			continue;
		def[nd].p = bs;
		def[nd].n = nn;
		def[nd].sq = best;
		def[nd].fc = bf;
		def[nd].t = idx[k];
		nd++;
	}
	meshFlushDeferred(M, def, nd, C, r, P);
}

PXH_D void meshPoly(const MeshSet& M, const int* idx, int nc, const Poly& H, const xf& pose, float cd, MPatches& P)
{
	const m33 R = qmat(pose.q);
	for (int k = 0; k < nc; k++)
	{
		const MeshTri t = meshTri(M, idx[k]);
		if (meshCulled(t, pose.p))
			continue;
		int f = 0;
		float best = 3.402823466e+38f;
		for (int j = 0; j < H.np; j++)
		{
			const float d = dot(mmul(R, H.pn(j)), t.n);
			if (best > d) { best = d; f = j; }
		}
		f3 buf0[64 + 3], buf1[64 + 3];
		int n0 = H.pcount(f) > 64 ? 64 : H.pcount(f);
		for (int j = 0; j < n0; j++)
			buf0[j] = mmul(R, H.vert(H.pvert(f, j))) + pose.p;
		f3 m[3];
		meshPrism(t, m);
		f3* in = buf0;
		f3* out = buf1;
		for (int e = 0; e < 3 && n0 > 0; e++)
		{
			int n1 = 0;
			for (int j = 0; j < n0; j++)
			{
				const f3 a = in[j], b = in[(j + 1) % n0];
				const float da = dot(m[e], a - t.v[e]), db = dot(m[e], b - t.v[e]);
				if (da >= 0.0f)
					out[n1++] = a;
				if ((da >= 0.0f) != (db >= 0.0f))
					out[n1++] = a + (b - a) * (da / (da - db));
			}
			f3* tmp = in;
			in = out;
			out = tmp;
			n0 = n1;
		}
		for (int j = 0; j < n0; j++)
		{
			const float s = dot(in[j] - t.v[0], t.n);
			if (cd > s)
				meshAdd(P, t.n, in[j] - t.n * s, s);
		}
		int vbest = 0;
		float dbest = 3.402823466e+38f;
		for (int j = 0; j < H.nv; j++)
		{
			const float d = dot(mmul(R, H.vert(j)), t.n);
			if (dbest > d) { dbest = d; vbest = j; }
		}
		const f3 sv = mmul(R, H.vert(vbest)) + pose.p;
		if (dot(m[0], sv - t.v[0]) >= 0.0f && dot(m[1], sv - t.v[1]) >= 0.0f && dot(m[2], sv - t.v[2]) >= 0.0f)
		{
			const float s = dot(sv - t.v[0], t.n);
			if (cd > s)
				meshAdd(P, t.n, sv - t.n * s, s);
		}
	}
}

// ---------------------------------------------------------------------------
// One wave per body. The lane forms above spend a body's time in one lane: tree
// nodes, triangles and points one after the other, patches, clipped polygons and
// caches in scratch memory. Here the wave reads 64 tree nodes at a time and walks
// them in registers, its lanes take a triangle each (spheres, capsules; four
// lanes a triangle for polytopes, clipped in LDS), and the patches lie in
// registers, a point a lane. Points are added in the lane forms' order, so the
// contacts are the same. 2,116 bodies on a mesh: 275 us in lanes (a wave each), 34 so,
// the slowest body's chain of triangles and points.
// ---------------------------------------------------------------------------
constexpr int MESH_ROUND = 16;       // triangles clipped at a time
constexpr int MESH_CLIP = 24;        // vertices a clipped polygon may have here (longer ones: lane form)

struct MeshLds
{
	int found[MESH_MAX_TRIS], idx[MESH_MAX_TRIS];
	float4 pts[MESH_ROUND * (MESH_CLIP + 1)], tmp[MESH_ROUND * (MESH_CLIP + 1)];
};

PXH_D int firstLane(uint64_t m) { return __ffsll((unsigned long long)m) - 1; }

// MPatches over the wave: lane 9 k + j holds point j of patch k, the 9 lanes of a
// patch its normal, count and least separation. Every lane makes each call.
struct MeshWave
{
	f3 n, p;
	float maxPen, s;
	int count, np, patch, slot;

	PXH_D void init(int lane)
	{
		n = p = mk(0.0f, 0.0f, 0.0f);
		maxPen = s = 0.0f;
		count = np = 0;
		patch = lane / (MESH_PC + 1);
		slot = lane - patch * (MESH_PC + 1);
	}

	// meshReduce4 of the patch at lanes base ...: its count
	PXH_D int reduce4(int base, int cnt)
	{
		if (cnt <= 4)
			return cnt;
		int i0 = 0, i1 = -1, i2 = -1, i3 = -1;
		float best = laneOf(s, base);
		for (int i = 1; i < cnt; i++)
		{
			const float v = laneOf(s, base + i);
			if (best > v) { best = v; i0 = i; }
		}
		const f3 c0 = laneOf(p, base + i0), w = p - c0;
		const float dd = dot(w, w);
		best = -1.0f;
		for (int i = 0; i < cnt; i++)
		{
			const float v = laneOf(dd, base + i);
			if (i != i0 && v > best) { best = v; i1 = i; }
		}
		const f3 ax = cross(laneOf(p, (base + i1) & 63) - c0, laneOf(n, base));
		const float h = dot(w, ax);
		float mx = -3.402823466e+38f, mn = 3.402823466e+38f;
		for (int i = 0; i < cnt; i++)
		{
			if (i == i0 || i == i1) continue;
			const float v = laneOf(h, base + i);
			if (v > mx) { mx = v; i2 = i; }
			if (mn > v) { mn = v; i3 = i; }
		}
		if (i3 == i2 || mx * mn > 0.0f)
		{
			mx = -3.402823466e+38f;
			i3 = -1;
			for (int i = 0; i < cnt; i++)
			{
				if (i == i0 || i == i1 || i == i2) continue;
				const float v = laneOf(h, base + i);
				if (v > mx) { mx = v; i3 = i; }
			}
		}
		const int from = (base + (slot == 0 ? i0 : slot == 1 ? i1 : slot == 2 ? i2 : i3)) & 63;
		const f3 q = mk(__shfl(p.x, from), __shfl(p.y, from), __shfl(p.z, from));
		const float qs = __shfl(s, from);
		if (patch * (MESH_PC + 1) == base && slot < 4)
		{
			p = q;
			s = qs;
		}
		return 4;
	}

	// meshAdd
	PXH_D void add(int lane, f3 pn, f3 pp, float ps)
	{
		const uint64_t m = __ballot(patch < np && dot(n, pn) > 0.996f);
		if (m != 0ull)
		{
			const int base = firstLane(m), cnt = laneOf(count, base);
			const bool mine = patch * (MESH_PC + 1) == base;
			const f3 d = p - pp;
			const uint64_t same = __ballot(mine && slot < cnt && 1e-10f > dot(d, d));
			if (mine && maxPen > ps)
				maxPen = ps;
			if (same != 0ull)
			{
				if (lane == firstLane(same) && s > ps)
				{
					p = pp;
					s = ps;
				}
				return;
			}
			if (lane == base + cnt)
			{
				p = pp;
				s = ps;
			}
			const int now = cnt + 1 > MESH_PC ? reduce4(base, cnt + 1) : cnt + 1;
			if (mine)
				count = now;
			return;
		}
		int k = np;
		if (k == MESH_NPATCH)
		{
			k = 0;
			float most = laneOf(maxPen, 0);
			for (int j = 1; j < MESH_NPATCH; j++)
			{
				const float v = laneOf(maxPen, j * (MESH_PC + 1));
				if (v > most) { most = v; k = j; }
			}
			if (!(most > ps))
				return;
		}
		else
			np++;
		if (patch == k)
		{
			n = pn;
			count = 1;
			maxPen = ps;
			if (slot == 0)
			{
				p = pp;
				s = ps;
			}
		}
	}
};

// Candidate triangles of the bounds mn, mx in L.idx in triangle order; their
// number, more than MESH_MAX_TRIS when they don't fit
PXH_D int meshCandidates(const MeshSet& M, int root, int nodes, f3 mn, f3 mx, MeshLds& L, int lane)
{
	const int end = root + nodes;
	int nc = 0;
	for (int nd = root; nd < end;)
	{
		const int at = nd + lane < end ? nd + lane : end - 1;
		const float4 lo = M.nodeLo[at], hi = M.nodeHi[at];
		const int4 info = M.nodeInfo[at];
		const bool hit = !(lo.x > mx.x || mn.x > hi.x || lo.y > mx.y || mn.y > hi.y || lo.z > mx.z || mn.z > hi.z);
		const int next = hit ? at + 1 : info.z;
		uint64_t seen = 0;
		const int first = nd;
		while (nd < end && nd - first < 64)
		{
			seen |= 1ull << (nd - first);
			nd = laneOf(next, nd - first);
		}
		const bool leaf = hit && ((seen >> lane) & 1ull) != 0ull;
		for (int j = 0; __any(leaf && j < info.y); j++)
		{
			bool in = leaf && j < info.y;
			int t = 0;
			if (in)
			{
				t = M.leafTri[info.x + j];
				const float4 tl = M.lo[t], th = M.hi[t];
				in = !(tl.x > mx.x || mn.x > th.x || tl.y > mx.y || mn.y > th.y || tl.z > mx.z || mn.z > th.z);
			}
			const uint64_t m = __ballot(in);
			const int to = nc + int(__popcll(m & ((1ull << lane) - 1ull)));
			if (in && to < MESH_MAX_TRIS)
				L.found[to] = t;
			nc += int(__popcll(m));
			if (nc > MESH_MAX_TRIS)
				return nc;
		}
	}
	waveSync();
	for (int i = lane; i < nc; i += 64)
	{
		const int x = L.found[i];
		int rank = 0;
		for (int j = 0; j < nc; j++)
			rank += L.found[j] < x;
		L.idx[rank] = x;
	}
	waveSync();
	return nc;
}

PXH_D bool meshSameEdge(int a, int b, int c, int d) { return (a == c && b == d) || (a == d && b == c); }

// meshSphere (p0 = p1 = c) and meshCapsule for up to 64 triangles, one a lane
template <bool CAPSULE>
PXH_D void meshRoundWave(const MeshSet& M, const int* idx, int nc, f3 p0, f3 p1, f3 c, float r, float cd, int lane,
                         MeshWave& P)
{
	const float infl = r + cd;
	int nf = 0, fc = TF_FACE;   // points on the face; deferred feature
	f3 f0 = c, f1 = c, dp = c, dn = c;
	float s0 = 0.0f, s1 = 0.0f, sq = 0.0f;
	bool later = false;
	const MeshTri t = meshTri(M, idx[lane < nc ? lane : 0]);
	if (lane < nc && !meshCulled(t, c))
	{
		if (!CAPSULE)
		{
			f3 cp;
			sq = meshPointTri(c, t.v[0], t.v[1], t.v[2], cp, fc);
			if (infl * infl > sq)
			{
				if (fc == TF_FACE)
				{
					nf = 1;
					f0 = c - t.n * r;
					s0 = sqrtf(sq) - r;
				}
				else
				{
					later = true;
					dp = c;
					dn = normalize(c - cp);
				}
			}
		}
		else
		{
			f3 m[3];
			meshPrism(t, m);
			float t0 = 0.0f, t1 = 1.0f;
			bool empty = false;
#pragma unroll
			for (int e = 0; e < 3; e++)
			{
				const float a = dot(m[e], p0 - t.v[e]), b = dot(m[e], p1 - t.v[e]);
				if (empty)
					continue;
				if (0.0f > a && 0.0f > b)
					empty = true;
				else if (0.0f > a)
				{
					const float u = a / (a - b);
					if (u > t0) t0 = u;
				}
				else if (0.0f > b)
				{
					const float u = a / (a - b);
					if (t1 > u) t1 = u;
				}
			}
			if (!empty && t1 >= t0)
			{
				const f3 d = p1 - p0;
				const f3 q0 = p0 + d * t0, q1 = p0 + d * t1;
				const float h0 = dot(q0 - t.v[0], t.n), h1 = dot(q1 - t.v[0], t.n);
				if (infl > h0)
				{
					nf = 1;
					f0 = q0 - t.n * r;
					s0 = h0 - r;
				}
				if (t1 > t0 && infl > h1)
				{
					f1 = q1 - t.n * r;
					s1 = h1 - r;
					if (nf == 0) { f0 = f1; s0 = s1; }
					nf++;
				}
			}
			else
			{
				float best = 3.402823466e+38f;
				f3 bs = p0, bt = p0;
#pragma unroll
				for (int e = 0; e < 3; e++)
				{
					f3 cs, ct;
					const float q = meshSegClosest(p0, p1, t.v[e], t.v[(e + 1) % 3], cs, ct);
					if (best > q)
					{
						best = q;
						bs = cs;
						bt = ct;
						fc = e == 0 ? TF_E01 : e == 1 ? TF_E12 : TF_E20;
					}
				}
				if (best == 3.402823466e+38f)
					fc = TF_E01;
				if (infl * infl > best && best > 0.0f)
				{
					dn = normalize(bs - bt);
					later = dot(dn, t.n) > 0.0f;
					dp = bs;
					sq = best;
				}
			}
		}
	}
	const uint64_t face = __ballot(nf > 0), defer = __ballot(later);
	for (uint64_t m = face; m != 0ull; m &= m - 1ull)
	{
		const int l = firstLane(m);
		const f3 tn = laneOf(t.n, l);
		P.add(lane, tn, laneOf(f0, l), laneOf(s0, l));
		if (CAPSULE && laneOf(nf, l) == 2)
			P.add(lane, tn, laneOf(f1, l), laneOf(s1, l));
	}
	// deferred contacts by distance, each unless its edge or vertex is one of a
	// face contact's triangle or of an earlier deferred one's (or of its own
	// triangle twice)
	const int x0 = t.vi[0], x1 = t.vi[1], x2 = t.vi[2];
	const bool onVertex = fc == TF_V0 || fc == TF_V1 || fc == TF_V2;
	const int fa = fc == TF_V0 || fc == TF_E01 ? x0 : fc == TF_V1 || fc == TF_E12 ? x1 : x2;
	const int fb = fc == TF_E01 ? x1 : fc == TF_E12 ? x2 : x0;
	bool held = onVertex ? (fc == TF_V1 && x1 == x0) || (fc == TF_V2 && (x2 == x0 || x2 == x1))
	                     : (fc != TF_E01 && meshSameEdge(fa, fb, x0, x1)) ||
	                           (fc != TF_E01 && fc != TF_E12 && meshSameEdge(fa, fb, x1, x2));
	int rank = 0;
	for (uint64_t m = face | defer; m != 0ull; m &= m - 1ull)
	{
		const int l = firstLane(m);
		const int o0 = laneOf(x0, l), o1 = laneOf(x1, l), o2 = laneOf(x2, l);
		const float osq = laneOf(sq, l);
		const bool isFace = ((face >> l) & 1ull) != 0ull;
		const bool before = osq < sq || (osq == sq && l < lane);
		const bool has = onVertex ? fa == o0 || fa == o1 || fa == o2
		                          : meshSameEdge(fa, fb, o0, o1) || meshSameEdge(fa, fb, o1, o2) || meshSameEdge(fa, fb, o2, o0);
		rank += !isFace && before;
		held |= has && (isFace || before);
	}
	const f3 at = dp - dn * r;
	const float sep = sqrtf(sq) - r;
	const int nd = int(__popcll(defer));
	for (int i = 0; i < nd; i++)
	{
		const uint64_t m = __ballot(later && !held && rank == i);
		if (m == 0ull)
			continue;
		const int l = firstLane(m);
		P.add(lane, laneOf(dn, l), laneOf(at, l), laneOf(sep, l));
	}
}

// meshPoly, MESH_ROUND triangles at a time; false where a polygon grows past
// MESH_CLIP vertices
PXH_D bool meshPolyWave(const MeshSet& M, int nc, const Poly& H, const xf& pose, float cd, MeshLds& L, int lane,
                        MeshWave& P)
{
	const m33 R = qmat(pose.q);
	const int tri = lane >> 2, sub = lane & 3;
	float4* const pts = L.pts + tri * (MESH_CLIP + 1);
	float4* const tmp = L.tmp + tri * (MESH_CLIP + 1);
	for (int k0 = 0; k0 < nc; k0 += MESH_ROUND)
	{
		const int k = k0 + tri;
		const MeshTri t = meshTri(M, L.idx[k < nc ? k : nc - 1]);
		const bool live = k < nc && !meshCulled(t, pose.p);
		int f = 0x7FFFFFFF, vbest = 0x7FFFFFFF;
		float best = 3.402823466e+38f, dbest = best;
		for (int j = sub; j < H.np; j += 4)
		{
			const float d = dot(mmul(R, H.pn(j)), t.n);
			if (best > d) { best = d; f = j; }
		}
		for (int j = sub; j < H.nv; j += 4)
		{
			const float d = dot(mmul(R, H.vert(j)), t.n);
			if (dbest > d) { dbest = d; vbest = j; }
		}
		for (int off = 1; off < 4; off <<= 1)
		{
			const float ob = __shfl_xor(best, off), od = __shfl_xor(dbest, off);
			const int of = __shfl_xor(f, off), ov = __shfl_xor(vbest, off);
			if (ob < best || (ob == best && of < f)) { best = ob; f = of; }
			if (od < dbest || (od == dbest && ov < vbest)) { dbest = od; vbest = ov; }
		}
		if (f == 0x7FFFFFFF) f = 0;
		if (vbest == 0x7FFFFFFF) vbest = 0;
		f3 m[3];
		meshPrism(t, m);
		const int corners = H.pcount(f);
		bool fits = corners <= MESH_CLIP;
		if (live && fits)
			for (int j = sub; j < corners; j += 4)
				tmp[j] = f4(mmul(R, H.vert(H.pvert(f, j))) + pose.p, 0.0f);
		waveSync();
		int n0 = 0;
		if (live && fits && sub == 0)
		{
			n0 = corners;
#pragma unroll
			for (int e = 0; e < 3; e++)
			{
				const float4* const in = e == 1 ? pts : tmp;
				float4* const out = e == 1 ? tmp : pts;
				int n1 = 0;
				f3 a = mk(in[0]);
				float da = dot(m[e], a - t.v[e]);
				const f3 a0 = a;
				const float d0 = da;
				for (int j = 0; j < n0; j++)
				{
					const bool last = j + 1 == n0;
					const f3 b = last ? a0 : mk(in[j + 1]);
					const float db = last ? d0 : dot(m[e], b - t.v[e]);
					if (da >= 0.0f)
					{
						if (n1 < MESH_CLIP) out[n1] = f4(a, 0.0f);
						n1++;
					}
					if ((da >= 0.0f) != (db >= 0.0f))
					{
						if (n1 < MESH_CLIP) out[n1] = f4(a + (b - a) * (da / (da - db)), 0.0f);
						n1++;
					}
					a = b;
					da = db;
				}
				fits &= n1 <= MESH_CLIP;
				n0 = n1 <= MESH_CLIP ? n1 : 0;
			}
			int keep = 0;
			for (int j = 0; j < n0; j++)
			{
				const f3 a = mk(pts[j]);
				const float s = dot(a - t.v[0], t.n);
				if (cd > s)
					pts[keep++] = f4(a - t.n * s, s);
			}
			const f3 sv = mmul(R, H.vert(vbest)) + pose.p;
			if (dot(m[0], sv - t.v[0]) >= 0.0f && dot(m[1], sv - t.v[1]) >= 0.0f && dot(m[2], sv - t.v[2]) >= 0.0f)
			{
				const float s = dot(sv - t.v[0], t.n);
				if (cd > s)
					pts[keep++] = f4(sv - t.n * s, s);   // one past MESH_CLIP at most
			}
			n0 = keep;
		}
		if (__any(live && !fits))
			return false;
		waveSync();
		for (uint64_t w = __ballot(n0 > 0); w != 0ull; w &= w - 1ull)
		{
			const int l = firstLane(w), cnt = laneOf(n0, l);
			const f3 tn = laneOf(t.n, l);
			for (int j = 0; j < cnt; j++)
			{
				const float4 q = L.pts[(l >> 2) * (MESH_CLIP + 1) + j];
				P.add(lane, tn, mk(q), q.w);
			}
		}
		waveSync();
	}
	return true;
}

}  // namespace pxh
