// Convex contact generation on the device: convex mesh (and the box seen as a
// polytope) against convex mesh, sphere, capsule and plane. The support steps that
// drop pairs take eight lanes a pair (convexApart), the separation search a wave
// (convexSeparationWave; one lane for hulls past its LDS, polySeparation), the
// contacts of hull pairs 16 lanes (convexContactsGroup), those of spheres, capsules
// and planes against a hull a wave, capsules against a box a lane (capsulePoly).
// Each generator follows the reference's PCM contact generation on a fresh
// manifold, so a pair gives the contacts of PxGenerateContacts with an empty
// PxCache: the separation is the exact closest-feature distance or minimum
// translation (what the reference's GJK / EPA converge to on polytopes), the
// witness polygons, polygon clipping and reduction to four points follow
// geomutils/src/pcm/GuPCMContactGenBoxConvex.cpp and GuPCMContactGenUtil.cpp.
#pragma once
#include "pxh_kernels.h"
#include "pxh_np.h"

namespace pxh {

constexpr int GEOM_CONVEXMESH = 5;
constexpr int HULL_MAX_POLY_VERTS = 16;   // polygon size the device path accepts
constexpr int HULL_MAX_CONTACTS = 32;     // clipped points before reduction

// PCMPolygonalBox (geomutils/src/pcm/GuPCMShapeConvex.cpp:40-136): the quads
// of gPCMBoxPolygonData, their planes, and the box's edges in polygon order
__constant__ const uint8_t kBoxQuads[24] = {0, 3, 2, 1, 1, 2, 6, 5, 5, 6, 7, 4, 4, 7, 3, 0, 3, 7, 6, 2, 4, 0, 1, 5};
__constant__ const uint32_t kBoxEdges[12] = {0x03000300u, 0x04000203u, 0x01000102u, 0x05000001u,
                                             0x04010602u, 0x02010506u, 0x05010105u, 0x04020706u,
                                             0x03020407u, 0x05020504u, 0x04030307u, 0x05030400u};

// One polytope: a hull (its arrays, in global memory or staged in LDS), or a
// box by its half extents.
struct Poly
{
	const float4* v;         // vertices
	const float4* pl;        // planes
	const uint32_t* poly;    // first vref | count << 16
	const uint8_t* vr;       // vertex loops
	const uint32_t* ed;      // edges
	int nv, np, ne;
	bool box;
	f3 h;
	float margin;
	float slack;   // how far polygon vertices lie below their planes
	float radius;  // of the vertices about the origin

	PXH_D f3 vert(int i) const
	{
		if (box)
			return mk((i == 1 || i == 2 || i == 5 || i == 6) ? h.x : -h.x,
			          (i == 2 || i == 3 || i == 6 || i == 7) ? h.y : -h.y, i >= 4 ? h.z : -h.z);
		return mk(v[i]);
	}
	PXH_D f3 pn(int f) const
	{
		if (box)
		{
			const float s = (f == 1 || f == 2 || f == 4) ? 1.0f : -1.0f;
			return (f == 1 || f == 3) ? mk(s, 0.0f, 0.0f) : ((f == 4 || f == 5) ? mk(0.0f, s, 0.0f) : mk(0.0f, 0.0f, s));
		}
		return mk(pl[f]);
	}
	PXH_D float pd(int f) const
	{
		if (box)
			return (f == 1 || f == 3) ? -h.x : ((f == 4 || f == 5) ? -h.y : -h.z);
		return pl[f].w;
	}
	PXH_D int pcount(int f) const { return box ? 4 : int(poly[f] >> 16); }
	PXH_D int pvert(int f, int k) const
	{
		return box ? int(kBoxQuads[4 * f + k]) : int(vr[int(poly[f] & 0xFFFFu) + k]);
	}
	PXH_D uint32_t edge(int e) const { return box ? kBoxEdges[e] : ed[e]; }
};

PXH_D Poly hullPoly(const HullSet& hs, int id)
{
	Poly p;
	const int4 a = hs.info[id], b = hs.info2[id];
	p.v = hs.v + a.x;
	p.pl = hs.pl + a.z;
	p.poly = hs.poly + a.z;
	p.vr = hs.vr + b.x;
	p.ed = hs.edge + b.y;
	p.nv = a.y; p.np = a.w; p.ne = b.z;
	p.box = false;
	p.h = mk(0.0f, 0.0f, 0.0f);
	p.margin = hs.bc[id].w;
	p.slack = __int_as_float(b.w);
	p.radius = hs.be[id].w;
	return p;
}

// BoxV margin: 15% of the smallest half extent (geomutils/src/gjk/GuVecBox.h:46, :56-75)
PXH_D Poly boxPoly(f3 h)
{
	Poly p;
	p.v = p.pl = nullptr;
	p.poly = p.ed = nullptr;
	p.vr = nullptr;
	p.nv = 8; p.np = 6; p.ne = 12;
	p.box = true;
	p.h = h;
	p.margin = fminf(h.x, fminf(h.y, h.z)) * 0.15f;
	p.slack = 0.0f;
	p.radius = sqrtf(dot(h, h));
	return p;
}

PXH_D f3 mxtransinv(const mxf& t, f3 v) { return mtmul(t.r, v - t.p); }
PXH_D mxf mxfOf(const xf& t) { mxf m; m.r = qmat(t.q); m.p = t.p; return m; }

// a point of polygon f's plane inside its counter-clockwise loop
PXH_D bool inPolygon(const Poly& P, int f, f3 q)
{
	const f3 n = P.pn(f);
	const int c = P.pcount(f);
	for (int k = 0; k < c; k++)
	{
		const f3 a = P.vert(P.pvert(f, k)), b = P.vert(P.pvert(f, (k + 1) % c));
		if (dot(q - a, cross(b - a, n)) > 0.0f)
			return false;
	}
	return true;
}

// closest points of segments p1q1, p2q2 (Ericson, Real-Time Collision
// Detection, 5.1.9); returns the squared distance
PXH_D float segClosestSq(f3 p1, f3 q1, f3 p2, f3 q2, f3& c1, f3& c2)
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

// Separation of A (placed in B's frame by aToB) and B. A face axis that
// separates them by more than cd ends the search (no contact possible; dist
// is that separation). Separated: exact
// closest points, dist > 0, n = (cA - cB) / dist. Overlapping: the minimum
// translation over both polytopes' face normals and the edge pairs that form
// a face of the Minkowski difference (their arcs cross on the Gauss maps;
// Gregorius, "The Separating Axis Test between Convex Polyhedra", GDC 2013);
// dist = -depth, n from B towards A.
PXH_D void polySeparation(const Poly& A, const mxf& aToB, const Poly& B, float cd, float& dist, f3& n, f3& cA,
                           f3& cB)
{
	float best = FLT_BIG;
	bool sep = false;
	for (int f = 0; f < B.np && !sep; f++)
	{
		const f3 bn = B.pn(f);
		const float bd = B.pd(f);
		float mn = FLT_BIG;
		f3 vmin = mk(0.0f, 0.0f, 0.0f);
		for (int i = 0; i < A.nv; i++)
		{
			const f3 va = mxtrans(aToB, A.vert(i));
			const float h = dot(bn, va) + bd;
			if (h < mn) { mn = h; vmin = va; }
		}
		if (mn > cd)
		{
			dist = mn;   // farther apart than the contact distance along this axis
			return;
		}
		if (mn > 0.0f) sep = true;
		else if (-mn < best)
		{
			best = -mn;
			n = bn;
			cA = vmin;
			cB = vmin - bn * mn;
		}
	}
	for (int f = 0; f < A.np && !sep; f++)
	{
		const f3 an = mmul(aToB.r, A.pn(f));
		const float ad = A.pd(f) - dot(an, aToB.p);
		float mn = FLT_BIG;
		f3 vmin = mk(0.0f, 0.0f, 0.0f);
		for (int i = 0; i < B.nv; i++)
		{
			const f3 vb = B.vert(i);
			const float h = dot(an, vb) + ad;
			if (h < mn) { mn = h; vmin = vb; }
		}
		if (mn > cd)
		{
			dist = mn;
			return;
		}
		if (mn > 0.0f) sep = true;
		else if (-mn < best)
		{
			best = -mn;
			n = -an;
			cB = vmin;
			cA = vmin - an * mn;
		}
	}
	if (!sep)
	{
		f3 bmean = mk(0.0f, 0.0f, 0.0f);
		for (int i = 0; i < B.nv; i++)
			bmean = bmean + B.vert(i);
		bmean = bmean * (1.0f / float(B.nv));
		for (int ea = 0; ea < A.ne && !sep; ea++)
		{
			const uint32_t e = A.edge(ea);
			const f3 a0 = mxtrans(aToB, A.vert(int(e & 0xFF))), a1 = mxtrans(aToB, A.vert(int((e >> 8) & 0xFF)));
			const f3 na = mmul(aToB.r, A.pn(int((e >> 16) & 0xFF))), nb = mmul(aToB.r, A.pn(int(e >> 24)));
			const f3 bxa = cross(nb, na);
			for (int ebi = 0; ebi < B.ne && !sep; ebi++)
			{
				const uint32_t g = B.edge(ebi);
				const f3 nc = -B.pn(int((g >> 16) & 0xFF)), nd = -B.pn(int(g >> 24));
				const f3 dxc = cross(nd, nc);
				const float cba = dot(nc, bxa), dba = dot(nd, bxa), adc = dot(na, dxc), bdc = dot(nb, dxc);
				if (!(cba * dba < 0.0f && adc * bdc < 0.0f && cba * bdc > 0.0f))
					continue;
				const f3 b0 = B.vert(int(g & 0xFF)), b1 = B.vert(int((g >> 8) & 0xFF));
				f3 ax = cross(a1 - a0, b1 - b0);
				const float l2 = dot(ax, ax);
				if (l2 < 1e-12f)
					continue;
				ax = ax * (1.0f / sqrtf(l2));
				if (dot(ax, b0 - bmean) < 0.0f)
					ax = -ax;
				const float ov = dot(ax, b0) - dot(ax, a0);
				if (ov < 0.0f) sep = true;
				else if (ov < best)
				{
					f3 c1, c2;
					segClosestSq(a0, a1, b0, b1, c1, c2);
					best = ov;
					n = ax;
					cA = c1;
					cB = c2;
				}
			}
		}
	}
	if (!sep)
	{
		dist = -best;
		return;
	}
	float d2 = FLT_BIG;
	for (int f = 0; f < B.np; f++)
	{
		const f3 bn = B.pn(f);
		const float bd = B.pd(f);
		for (int i = 0; i < A.nv; i++)
		{
			const f3 va = mxtrans(aToB, A.vert(i));
			const float h = dot(bn, va) + bd;
			if (h < 0.0f || h * h >= d2)
				continue;
			const f3 q = va - bn * h;
			if (!inPolygon(B, f, q))
				continue;
			d2 = h * h; cA = va; cB = q;
		}
	}
	for (int f = 0; f < A.np; f++)
	{
		const f3 an = mmul(aToB.r, A.pn(f));
		const float ad = A.pd(f) - dot(an, aToB.p);
		for (int i = 0; i < B.nv; i++)
		{
			const f3 vb = B.vert(i);
			const float h = dot(an, vb) + ad;
			if (h < 0.0f || h * h >= d2)
				continue;
			const f3 q = vb - an * h;
			if (!inPolygon(A, f, mxtransinv(aToB, q)))
				continue;
			d2 = h * h; cB = vb; cA = q;
		}
	}
	for (int ea = 0; ea < A.ne; ea++)
	{
		const uint32_t e = A.edge(ea);
		const f3 a0 = mxtrans(aToB, A.vert(int(e & 0xFF))), a1 = mxtrans(aToB, A.vert(int((e >> 8) & 0xFF)));
		for (int ebi = 0; ebi < B.ne; ebi++)
		{
			const uint32_t g = B.edge(ebi);
			f3 c1, c2;
			const float s = segClosestSq(a0, a1, B.vert(int(g & 0xFF)), B.vert(int((g >> 8) & 0xFF)), c1, c2);
			if (s < d2) { d2 = s; cA = c1; cB = c2; }
		}
	}
	dist = sqrtf(d2);
	n = (cA - cB) * (1.0f / dist);
}

PXH_D void waveArgMin(float& v, uint32_t& idx);
PXH_D float waveMin(float v);
PXH_D f3 laneOf(f3 v, int l);
template <int LANES> PXH_D int witnessPolygonLanes(const Poly& P, f3 normal, f3 closest, float tolerance, int lane);

// Gu::getWitnessPolygonIndex (geomutils/src/pcm/GuPCMContactGenUtil.cpp:201-271);
// the per-polygon distances are evaluated again in the second pass
PXH_D int witnessPolygon(const Poly& P, f3 normal, f3 closest, float tolerance)
{
	const float eps = -tolerance;
	float dist = dot(P.pn(0), closest) + P.pd(0);
	float minDist = dist >= eps ? fabsf(dist) : FLT_BIG;
	float maxDist = dist;
	int maxIdx = 0, idx = 0;
	for (int i = 1; i < P.np; i++)
	{
		dist = dot(P.pn(i), closest) + P.pd(i);
		const float pdi = dist >= eps ? fabsf(dist) : FLT_BIG;
		if (minDist > pdi) { minDist = pdi; idx = i; }
		if (dist > maxDist) { maxDist = dist; maxIdx = i; }
	}
	if (minDist == FLT_BIG)
		return maxIdx;
	float bestProj = dot(normalize(P.pn(idx)), normal);
	const int first = idx;
	for (int i = 0; i < P.np; i++)
	{
		const float di = dot(P.pn(i), closest) + P.pd(i);
		const float pdi = di >= eps ? fabsf(di) : FLT_BIG;
		if ((tolerance > (pdi - minDist)) && (first != i))
		{
			const float proj = dot(normalize(P.pn(i)), normal);
			if (bestProj > proj) { idx = i; bestProj = proj; }
		}
	}
	return idx;
}

// Gu::findRotationMatrixFromZAxis (geomutils/src/pcm/GuPersistentContactManifold.cpp:289-354):
// a rotation whose third row is `to`
PXH_D m33 rotFromZ(f3 to)
{
	m33 m;
	const float e = to.z, f = fabsf(e);
	if (0.9999f > f)
	{
		const float vx = -to.y, vy = to.x;
		const float h = 1.0f / (1.0f + e);
		const float hvx = h * vx, hvxy = hvx * vy;
		m.c0 = mk(hvx * vx + e, hvxy, vy);
		m.c1 = mk(hvxy, h * (vy * vy) + e, -vx);
		m.c2 = mk(-vy, vx, e);
		return m;
	}
	const f3 from = mk(0.0f, 0.0f, 1.0f), absFrom = mk(0.0f, 1.0f, 0.0f);
	const f3 u = absFrom - from, v = absFrom - to;
	const float du = dot(u, u), dv = dot(v, v), duv = dot(u, v);
	const float c1 = -(2.0f / du), c2 = -(2.0f / dv), c3 = c1 * (c2 * duv);
	const f3 c1u = u * c1, c2v = v * c2, c3v = v * c3;
	m.c0 = u * c1u.x + (v * c2v.x + u * c3v.x);
	m.c0.x += 1.0f;
	m.c1 = u * c1u.y + (v * c2v.y + u * c3v.y);
	m.c1.y += 1.0f;
	m.c2 = u * c1u.z + (v * c2v.z + u * c3v.z);
	m.c2.z += 1.0f;
	return m;
}

PXH_D float triArea2(f3 a, f3 b, f3 c)
{
	const f3 ca = a - c, cb = b - c;
	return ca.x * cb.y - ca.y * cb.x;
}

// Gu::contains (geomutils/src/pcm/GuPCMContactGenUtil.cpp:35-103) for an n-gon
template <class V> PXH_D bool polyContainsN(const V* verts, int nv, f3 p, f3 mn, f3 mx)
{
	if ((mn.x > p.x || p.x > mx.x) || (mn.y > p.y || p.y > mx.y))
		return false;
	const float tx = p.x, ty = p.y, eps = 1.1920928955078125e-7f;
	int inter = 0;
	for (int i = 0, j = nv - 1; i < nv; j = i++)
	{
		const float jy = verts[j].y, iy = verts[i].y, jx = verts[j].x, ix = verts[i].x;
		if ((tx == jx && ty == jy) || (tx == ix && ty == iy))
			return true;
		if ((jy > ty) != (iy > ty))
		{
			const float jix = ix - jx, jiy = iy - jy, jty = ty - jy;
			const float part1 = jty * jix, part2 = (jx + eps) * jiy, part3 = tx * jiy;
			const bool cmp = jiy > 0.0f;
			const float tmp = part1 + part2;
			if ((cmp ? tmp : part3) >= (cmp ? part3 : tmp))
			{
				if (inter == 1)
					return false;
				inter++;
			}
		}
	}
	return inter > 0;
}

// Gu::pcmContactSphereConvex on a fresh manifold
// (geomutils/src/pcm/GuPCMContactSphereConvex.cpp:110-246)
// (over the wave: the lanes share the faces and edges, the first minimum in
// their order wins)
PXH_D int sphereConvexWave(float r, f3 p0, const Poly& B, const xf& x1, float cd, int lane, Contacts& o)
{
	const f3 c = xtransinv(x1, p0);
	float least = FLT_BIG;   // minus the largest height
	uint32_t fm = 0xFFFFFFFFu;
	for (int f = lane; f < B.np; f += 64)
	{
		const float h = dot(B.pn(f), c) + B.pd(f);
		if (-h < least) { least = -h; fm = uint32_t(f); }
	}
	waveArgMin(least, fm);
	const float hmax = -least;
	f3 n;
	float pen;
	if (hmax <= 0.0f)
	{
		n = B.pn(fm == 0xFFFFFFFFu ? 0 : int(fm));
		pen = hmax - r;
	}
	else
	{
		float d2 = FLT_BIG;
		uint32_t at = 0xFFFFFFFFu;
		f3 q = c;
		for (int f = lane; f < B.np; f += 64)
		{
			const f3 bn = B.pn(f);
			const float h = dot(bn, c) + B.pd(f);
			if (h < 0.0f || h * h >= d2)
				continue;
			const f3 pq = c - bn * h;
			if (inPolygon(B, f, pq)) { d2 = h * h; q = pq; at = uint32_t(f); }
		}
		for (int e = lane; e < B.ne; e += 64)
		{
			const uint32_t g = B.edge(e);
			f3 c1, c2;
			const float s = segClosestSq(c, c, B.vert(int(g & 0xFF)), B.vert(int((g >> 8) & 0xFF)), c1, c2);
			if (s < d2) { d2 = s; q = c2; at = uint32_t(B.np + e); }
		}
		const uint32_t mine = at;
		waveArgMin(d2, at);
		const uint64_t m = __ballot(mine == at && at != 0xFFFFFFFFu);
		q = m ? laneOf(q, __ffsll((unsigned long long)m) - 1) : c;
		const float dist = sqrtf(d2);
		if (dist > r + cd)
			return 0;
		n = (c - q) * (1.0f / dist);
		pen = dist - r;
	}
	const f3 wn = qrot(x1.q, n);
	o.n = wn;
	o.p[0] = p0 - wn * r;
	o.sep[0] = pen;
	o.count = 1;
	return 1;
}

// Capsule core segment pq against polytope B (B's frame), standing in for
// GJK / EPA on the segment (geomutils/src/gjk/GuGJKPenetration.h:95-306 with
// takeCoreShape: points on the segment, distance without the radius). Apart:
// the exact closest points, returns dist > 0 with n = (cA - cB)/dist.
// Entering B: the minimum translation over B's face normals and the
// directions normal to the segment and each edge of B (the face normals of
// their Minkowski difference), returns -depth, cB = cA + n depth.
PXH_D float segPoly(const Poly& B, f3 p, f3 q, f3& n, f3& cA, f3& cB)
{
	const f3 d = q - p;
	float t0 = 0.0f, t1 = 1.0f;
	bool enters = true;
	cA = p;
	cB = p;
	for (int f = 0; f < B.np && enters; f++)
	{
		const f3 fn = B.pn(f);
		const float hp = dot(fn, p) + B.pd(f), dn = dot(fn, d);
		if (dn == 0.0f)
		{
			enters = !(hp > 0.0f);
			continue;
		}
		const float t = -hp / dn;
		if (dn < 0.0f)
			t0 = fmaxf(t0, t);
		else
			t1 = fminf(t1, t);
		enters = !(t0 > t1);
	}
	if (!enters)
	{
		float best = FLT_BIG;
		for (int k = 0; k < 2; k++)
		{
			const f3 c = k ? q : p;
			for (int f = 0; f < B.np; f++)
			{
				const f3 fn = B.pn(f);
				const float h = dot(fn, c) + B.pd(f);
				if (h < 0.0f || h * h >= best)
					continue;
				const f3 pc = c - fn * h;
				if (inPolygon(B, f, pc)) { best = h * h; cA = c; cB = pc; }
			}
		}
		for (int e = 0; e < B.ne; e++)
		{
			const uint32_t ed = B.edge(e);
			f3 c1, c2;
			const float s = segClosestSq(p, q, B.vert(ed & 0xFF), B.vert((ed >> 8) & 0xFF), c1, c2);
			if (s < best) { best = s; cA = c1; cB = c2; }
		}
		const float dist = sqrtf(best);
		n = (cA - cB) * (1.0f / dist);
		return dist;
	}
	float best = FLT_BIG;
	int bestEdge = -1;
	f3 axis = mk(1.0f, 0.0f, 0.0f);
	for (int f = 0; f < B.np; f++)
	{
		const f3 fn = B.pn(f);
		const float depth = -B.pd(f) - fminf(dot(fn, p), dot(fn, q));
		if (depth < best) { best = depth; axis = fn; }
	}
	for (int e = 0; e < B.ne; e++)
	{
		const uint32_t ed = B.edge(e);
		const f3 a = B.vert(ed & 0xFF), b = B.vert((ed >> 8) & 0xFF);
		f3 c = cross(d, b - a);
		const float l2 = dot(c, c);
		if (!(l2 > 1e-12f))
			continue;
		c = c * (1.0f / sqrtf(l2));
		float mnB = FLT_BIG, mxB = -FLT_BIG;
		for (int i = 0; i < B.nv; i++)
		{
			const float s = dot(c, B.vert(i));
			mnB = fminf(mnB, s);
			mxB = fmaxf(mxB, s);
		}
		const float sp = dot(c, p), sq = dot(c, q);
		const float dp = mxB - fminf(sp, sq), dm = fmaxf(sp, sq) - mnB;
		if (dp < best) { best = dp; axis = c; bestEdge = e; }
		if (dm < best) { best = dm; axis = -c; bestEdge = e; }
	}
	n = axis;
	if (bestEdge >= 0)
	{
		const uint32_t ed = B.edge(bestEdge);
		f3 c2;
		segClosestSq(p, q, B.vert(ed & 0xFF), B.vert((ed >> 8) & 0xFF), cA, c2);
	}
	else
		cA = dot(axis, q) < dot(axis, p) ? q : p;
	cB = cA + axis * best;
	return -best;
}

// whether some of B's planes keep the segment p, q outside, in one lane; the test
// that segPoly, segPolyWave and (p = q) sphereConvexWave take a contact inside by
PXH_D bool planesKeepOut(const Poly& B, f3 p, f3 q)
{
	const f3 d = q - p;
	float t0 = 0.0f, t1 = 1.0f;
	bool out = false;
	for (int f = 0; f < B.np && !out; f++)
	{
		const f3 fn = B.pn(f);
		const float hp = dot(fn, p) + B.pd(f), dn = dot(fn, d);
		if (dn == 0.0f)
			out = hp > 0.0f;
		else if (dn < 0.0f)
			t0 = fmaxf(t0, -hp / dn);
		else
			t1 = fminf(t1, -hp / dn);
		out |= t0 > t1;
	}
	return out;
}

// segPoly over the wave: the lanes share B's faces and edges, the first minimum
// in their order wins
PXH_D float segPolyWave(const Poly& B, f3 p, f3 q, int lane, f3& n, f3& cA, f3& cB)
{
	const f3 d = q - p;
	float t0 = 0.0f, t1 = 1.0f;
	bool out = false;
	for (int f = lane; f < B.np; f += 64)
	{
		const f3 fn = B.pn(f);
		const float hp = dot(fn, p) + B.pd(f), dn = dot(fn, d);
		if (dn == 0.0f)
			out |= hp > 0.0f;
		else if (dn < 0.0f)
			t0 = fmaxf(t0, -hp / dn);
		else
			t1 = fminf(t1, -hp / dn);
	}
	t0 = -waveMin(-t0);
	t1 = waveMin(t1);
	float best = FLT_BIG;
	uint32_t at = 0xFFFFFFFFu;
	cA = p;
	cB = p;
	if (__any(out) || t0 > t1)
	{
		for (int k = lane; k < 2 * B.np; k += 64)
		{
			const int f = k < B.np ? k : k - B.np;
			const f3 c = k < B.np ? p : q;
			const f3 fn = B.pn(f);
			const float h = dot(fn, c) + B.pd(f);
			if (h < 0.0f || h * h >= best)
				continue;
			const f3 pc = c - fn * h;
			if (inPolygon(B, f, pc)) { best = h * h; cA = c; cB = pc; at = uint32_t(k); }
		}
		for (int e = lane; e < B.ne; e += 64)
		{
			const uint32_t ed = B.edge(e);
			f3 c1, c2;
			const float s = segClosestSq(p, q, B.vert(ed & 0xFF), B.vert((ed >> 8) & 0xFF), c1, c2);
			if (s < best) { best = s; cA = c1; cB = c2; at = uint32_t(2 * B.np + e); }
		}
		const uint32_t mine = at;
		waveArgMin(best, at);
		const uint64_t m = __ballot(mine == at && at != 0xFFFFFFFFu);
		const int l = m ? __ffsll((unsigned long long)m) - 1 : 0;
		cA = m ? laneOf(cA, l) : p;
		cB = m ? laneOf(cB, l) : p;
		const float dist = sqrtf(best);
		n = (cA - cB) * (1.0f / dist);
		return dist;
	}
	f3 axis = mk(1.0f, 0.0f, 0.0f);
	for (int f = lane; f < B.np; f += 64)
	{
		const f3 fn = B.pn(f);
		const float depth = -B.pd(f) - fminf(dot(fn, p), dot(fn, q));
		if (depth < best) { best = depth; axis = fn; at = uint32_t(f); }
	}
	for (int e = lane; e < B.ne; e += 64)
	{
		const uint32_t ed = B.edge(e);
		const f3 a = B.vert(ed & 0xFF), b = B.vert((ed >> 8) & 0xFF);
		f3 c = cross(d, b - a);
		const float l2 = dot(c, c);
		if (!(l2 > 1e-12f))
			continue;
		c = c * (1.0f / sqrtf(l2));
		float mnB = FLT_BIG, mxB = -FLT_BIG;
		for (int i = 0; i < B.nv; i++)
		{
			const float s = dot(c, B.vert(i));
			mnB = fminf(mnB, s);
			mxB = fmaxf(mxB, s);
		}
		const float sp = dot(c, p), sq = dot(c, q);
		const float dp = mxB - fminf(sp, sq), dm = fmaxf(sp, sq) - mnB;
		if (dp < best) { best = dp; axis = c; at = uint32_t(B.np + e); }
		if (dm < best) { best = dm; axis = -c; at = uint32_t(B.np + e); }
	}
	const uint32_t mine = at;
	waveArgMin(best, at);
	const uint64_t m = __ballot(mine == at && at != 0xFFFFFFFFu);
	axis = m ? laneOf(axis, __ffsll((unsigned long long)m) - 1) : mk(1.0f, 0.0f, 0.0f);
	n = axis;
	if (at != 0xFFFFFFFFu && at >= uint32_t(B.np))
	{
		const uint32_t ed = B.edge(int(at) - B.np);
		f3 c2;
		segClosestSq(p, q, B.vert(ed & 0xFF), B.vert((ed >> 8) & 0xFF), cA, c2);
	}
	else
		cA = dot(axis, q) < dot(axis, p) ? q : p;
	cB = cA + axis * best;
	return -best;
}

constexpr int CAPSULE_MAX_CONTACTS = HULL_MAX_POLY_VERTS + 2;

// generatedCapsuleBoxFaceContacts (geomutils/src/pcm/GuPCMContactGenSphereCapsule.cpp:221-284):
// each endpoint moved along -n onto the reference polygon's plane, kept when
// that distance is within radius + contact distance and the foot lies in the
// polygon
PXH_D void capsuleFaceContacts(const Poly& B, int f, f3 p0, f3 p1, f3 n, float infl, const mxf& aToB, PC* mc, int& nc)
{
	const f3 pn = normalize(B.pn(f));
	const int nv = B.pcount(f);
	const f3 a = B.vert(B.pvert(f, 0));
	const float proj = dot(pn, n);
	const float numer = proj > 0.0f ? 1.0f / proj : 0.0f;
	const float t[2] = {dot(pn, p0 - a) * numer, dot(pn, p1 - a) * numer};
	if (!(infl >= t[0] || infl >= t[1]))
		return;
	const m33 rot = rotFromZ(pn);
	f3 pts[HULL_MAX_POLY_VERTS];
	f3 mn = mk(FLT_BIG, FLT_BIG, FLT_BIG), mx = -mn;
	for (int i = 0; i < nv; i++)
	{
		pts[i] = mmul(rot, B.vert(B.pvert(f, i)));
		mn = mk(fminf(mn.x, pts[i].x), fminf(mn.y, pts[i].y), fminf(mn.z, pts[i].z));
		mx = mk(fmaxf(mx.x, pts[i].x), fmaxf(mx.y, pts[i].y), fmaxf(mx.z, pts[i].z));
	}
	for (int k = 0; k < 2; k++)
	{
		if (!(infl >= t[k]))
			continue;
		const f3 e = k ? p1 : p0;
		const f3 foot = e - n * t[k];
		if (polyContainsN(pts, nv, mmul(rot, foot), mn, mx))
		{
			mc[nc].la = mxtransinv(aToB, e);
			mc[nc].lb = foot;
			mc[nc].ln = n;
			mc[nc].pen = t[k];
			nc++;
		}
	}
}

// intersectRayPolyhedron (GuPCMContactGenSphereCapsule.cpp:98-141): the entry
// parameter of the ray a + t dir, t >= 0, into B
PXH_D bool rayPolyhedronWave(const Poly& B, f3 a, f3 dir, int lane, float& tEnter)
{
	float tFirst = 0.0f, tLast = FLT_BIG;
	bool out = false;
	for (int k = lane; k < B.np; k += 64)
	{
		const f3 fn = B.pn(k);
		const float den = dot(fn, dir);
		const float dist = dot(fn, a) + B.pd(k);
		if (1e-7f > fabsf(den))
			out |= dist > 0.0f;
		else
		{
			const float t = -(dist / den);
			if (0.0f > den && t > tFirst)
				tFirst = t;
			if (!(0.0f > den) && tLast > t)
				tLast = t;
		}
	}
	tFirst = -waveMin(-tFirst);
	tLast = waveMin(tLast);
	tEnter = tFirst;
	return !(__any(out) || tFirst > tLast);
}

// generatedFaceContacts (GuPCMContactGenSphereCapsule.cpp:286-310): each
// endpoint's ray along -n into the hull, entered within radius + contact
// distance
PXH_D void capsuleRayContacts(const Poly& B, f3 p0, f3 p1, f3 n, float infl, const mxf& aToB, int lane, PC* mc, int& nc)
{
	for (int k = 0; k < 2; k++)
	{
		const f3 e = k ? p1 : p0;
		float tE;
		if (rayPolyhedronWave(B, e, -n, lane, tE) && infl >= tE)
		{
			mc[nc].la = mxtransinv(aToB, e);
			mc[nc].lb = (-n) * tE + e;
			mc[nc].ln = n;
			mc[nc].pen = tE;
			nc++;
		}
	}
}

// generateEE / generatedContactsEEContacts (GuPCMContactGenSphereCapsule.cpp:312-377):
// where the segment crosses the plane through a reference polygon edge
// spanned with n, a contact against that edge (its parameter within
// [-0.005, 1.005]) when the signed distance along n is within the radius
PXH_D void capsuleEEContacts(const Poly& B, int f, f3 p, f3 q, f3 normal, float infl, const mxf& aToB, PC* mc, int& nc)
{
	const int nv = B.pcount(f);
	for (int rs = 0, re = nv - 1; rs < nv; re = rs++)
	{
		const f3 a = B.vert(B.pvert(f, rs)), b = B.vert(B.pvert(f, re));
		const f3 ab = b - a;
		const f3 n = cross(ab, normal);
		const float d = dot(n, a);
		const float sp = dot(n, p) - d, sq = dot(n, q) - d;
		if (sp * sq > 0.0f)
			continue;
		const f3 pq = q - p;
		const float npq = dot(n, pq);
		if (npq == 0.0f)
			continue;
		const f3 lpa = pq * ((d - dot(n, p)) / npq) + p;
		const f3 perN = cross(normal, pq);
		const f3 ap = lpa - a;
		const float tv = dot(perN, ap) / dot(perN, ab);
		if (tv > 1.005f || -0.005f > tv)
			continue;
		const f3 v = ap - ab * tv;
		const float sd = dot(v, normal);
		if (infl >= sd)
		{
			mc[nc].la = mxtransinv(aToB, lpa);
			mc[nc].lb = lpa - v;
			mc[nc].ln = normal;
			mc[nc].pen = sd;
			nc++;
		}
	}
}

// PersistentContactManifold::reduceBatchContacts2
// (geomutils/src/pcm/GuPersistentContactManifold.cpp:1177-1243): the deepest
// point, the point farthest from it, then the last point (in order) of those
// nearer the second than the first that is shallower than the second
PXH_D void reduceBatch2(const PC* m, int n, int& i0, int& i1)
{
	int idx = 0;
	float maxD = m[0].pen;
	for (int i = 1; i < n; i++)
		if (maxD > m[i].pen) { maxD = m[i].pen; idx = i; }
	i0 = idx;
	const f3 b0 = m[i0].lb;
	f3 v = m[0].lb - b0;
	float far = dot(v, v);
	idx = 0;
	for (int i = 1; i < n; i++)
	{
		v = m[i].lb - b0;
		const float d = dot(v, v);
		if (d > far) { far = d; idx = i; }
	}
	const int first = idx;
	const float maxDepth = m[first].pen;
	const f3 b1 = m[first].lb;
	int second = first;
	for (int i = 0; i < n; i++)
	{
		if (i == i0 || i == first)
			continue;
		const f3 d0 = b0 - m[i].lb, d1 = b1 - m[i].lb;
		if (dot(d0, d0) > dot(d1, d1) && maxDepth > m[i].pen)
			second = i;
	}
	i1 = second;
}

// Gu::pcmContactCapsuleBox / pcmContactCapsuleConvex on a fresh manifold
// (geomutils/src/pcm/GuPCMContactCapsuleBox.cpp:42-200,
// GuPCMContactCapsuleConvex.cpp:43-236, full contact generation
// GuPCMContactGenSphereCapsule.cpp:379-468): the core segment against the
// polytope; box: endpoint contacts on the witness polygon, convex: endpoint
// rays into the hull; fewer than two: edge contacts on the witness polygon;
// none: the closest-point contact; reduced to two. Points on the capsule's
// surface, separation less the radius, normal from the polytope. BOX: one pair a
// lane; else a hull and one pair over the wave, every lane with the same points.
template <bool BOX>
PXH_D int capsulePoly(float r, float hh, const xf& x0, const Poly& B, const xf& x1, float cd, float tol, int lane,
                      Contacts& o)
{
	const mxf aToB = mxfOf(xinvmul(x1, x0));
	const f3 ext = mmul(aToB.r, mk(hh, 0.0f, 0.0f));
	const f3 p0 = aToB.p + ext, p1 = aToB.p - ext;
	f3 n, cA, cB;
	const float dist = BOX ? segPoly(B, p0, p1, n, cA, cB) : segPolyWave(B, p0, p1, lane, n, cA, cB);
	if (dist > r + cd)
		return 0;
	const float infl = r + cd;
	const float wtol = fminf(fmaxf(B.margin, tol * 1e-2f), tol * 5e-2f);
	PC mc[CAPSULE_MAX_CONTACTS];
	int nc = 0;
	if constexpr (BOX)
	{
		const int f = witnessPolygon(B, -n, cB, wtol);
		capsuleFaceContacts(B, f, p0, p1, n, infl, aToB, mc, nc);
		if (nc < 2)
			capsuleEEContacts(B, f, p0, p1, n, infl, aToB, mc, nc);
	}
	else
	{
		capsuleRayContacts(B, p0, p1, n, infl, aToB, lane, mc, nc);
		if (nc < 2)
			capsuleEEContacts(B, witnessPolygonLanes<64>(B, -n, cB, wtol, lane), p0, p1, n, infl, aToB, mc, nc);
	}
	int i0 = 0, i1 = 1;
	if (nc == 0)
	{
		mc[0].la = mxtransinv(aToB, cA);
		mc[0].lb = cB;
		mc[0].ln = n;
		mc[0].pen = dist;
		nc = 1;
	}
	else if (nc > 2)
	{
		reduceBatch2(mc, nc, i0, i1);
		nc = 2;
	}
	const f3 wn = qrot(x1.q, n);
	o.n = wn;
	o.count = 0;
	for (int i = 0; i < nc; i++)
	{
		const PC& c = mc[i == 0 ? i0 : i1];
		const float sep = c.pen - r;
		if (cd >= sep)
			pushContact(o, xtrans(x0, c.la) - wn * r, sep);
	}
	return o.count;
}

}  // namespace pxh

namespace pxh {

// ---------------------------------------------------------------------------
// One wavefront per convex pair: the 64 lanes split the face-axis, edge-pair
// and closest-feature searches of polySeparation over the pair's vertices,
// planes and edges staged in LDS. Every search keeps polySeparation's order
// (the first minimum in loop order wins), so the result is the same as the
// per-lane path's.
// ---------------------------------------------------------------------------
constexpr int CVX_WAVE_V = 64, CVX_WAVE_P = 128, CVX_WAVE_E = 192, CVX_ARCS = 32;

struct CvxLds
{
	float4 va[CVX_WAVE_V];   // A's vertices in B's frame
	float4 vb[CVX_WAVE_V];   // B's vertices
	float4 pa[CVX_WAVE_P];   // A's planes in B's frame
	float4 pb[CVX_WAVE_P];   // B's planes
	uint32_t ea[CVX_WAVE_E];
	uint32_t eb[CVX_WAVE_E];
	union
	{
		struct   // closest features of separated polytopes
		{
			uint32_t polyA[CVX_WAVE_P], polyB[CVX_WAVE_P];
			uint8_t vrA[2 * CVX_WAVE_E], vrB[2 * CVX_WAVE_E];   // a closed polytope has 2 vrefs per edge
			uint8_t elA[CVX_WAVE_E], elB[CVX_WAVE_E];           // vertices and edges that may hold them
		};
		struct   // edge pairs of overlapping ones
		{
			float4 arc[3 * CVX_ARCS];   // arcs of some of B's edges: both (negated) normals and their cross product
			uint32_t open[128];         // pairs whose arcs cross
		};
	};
};

PXH_D bool fitsWave(const Poly& A, const Poly& B)
{
	return A.nv <= CVX_WAVE_V && B.nv <= CVX_WAVE_V && A.np <= CVX_WAVE_P && B.np <= CVX_WAVE_P &&
	       A.ne <= CVX_WAVE_E && B.ne <= CVX_WAVE_E;
}

// LDS written by some lanes of the wave becomes visible to the others
PXH_D void waveSync()
{
	__builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
	__builtin_amdgcn_wave_barrier();
}

// smallest value over the wave, the lowest order index among equal values
PXH_D void waveArgMin(float& v, uint32_t& idx)
{
	for (int off = 32; off >= 1; off >>= 1)
	{
		const float ov = __shfl_xor(v, off);
		const uint32_t oi = __shfl_xor(idx, off);
		if (ov < v || (ov == v && oi < idx))
		{
			v = ov;
			idx = oi;
		}
	}
}

PXH_D bool waveAny(bool b) { return __ballot(b) != 0ull; }

PXH_D f3 ldsV(const float4* a, int i) { return mk(a[i].x, a[i].y, a[i].z); }

// (i, j) of the flat index k = i * n + j as a lane walks k = lane, lane + 64,
// ...: one division up front, then a step of 64 costs an add and one compare
// (a runtime integer division is a long instruction sequence on this target).
struct FlatPair
{
	int n, q, r, i, j;
	PXH_D FlatPair(int lane, int n_) : n(n_ > 0 ? n_ : 1)
	{
		q = 64 / n;
		r = 64 - q * n;
		i = lane / n;
		j = lane - i * n;
	}
	PXH_D void next()
	{
		i += q;
		j += r;
		if (j >= n)
		{
			j -= n;
			i++;
		}
	}
};

// True only if A and B are farther apart than need: Gilbert's iteration for the
// point of A - B nearest the origin (Gilbert 1966, "An iterative procedure for
// computing the minimum of a quadratic form on a convex set"), each step's
// support an axis that either shows the gap or moves v nearer. Eight lanes of a
// wave share a pair and hold the same v; lane sub has every eighth vertex in
// B's frame, the first 4 of each polytope in registers (a step reads no memory
// below 33 vertices).
constexpr int APART_LANES = 8, APART_ROUNDS = 8, APART_HELD = 4;

// the smallest h of 8 lanes and, from its lane (the lowest among equals), p
PXH_D void groupMin(float& h, f3& p)
{
	const int lane = __lane_id();
	float m = h;
	m = fminf(m, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(m), 0xB1, 0xF, 0xF, true)));    // quad 1 0 3 2
	m = fminf(m, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(m), 0x4E, 0xF, 0xF, true)));    // quad 2 3 0 1
	m = fminf(m, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(m), 0x141, 0xF, 0xF, true)));   // half-row mirror
	const uint32_t mine = uint32_t(__ballot(h == m) >> (lane & 56)) & 0xFFu;
	const int from = (lane & 56) + (mine ? __ffs(int(mine)) - 1 : 0);
	p = mk(__shfl(p.x, from), __shfl(p.y, from), __shfl(p.z, from));
	h = m;
}

PXH_D bool convexApart(const Poly& A, const mxf& aToB, const Poly& B, float need, int sub)
{
	f3 va[APART_HELD], vb[APART_HELD];
#pragma unroll
	for (int k = 0; k < APART_HELD; k++)
	{
		// past the last vertex: the first again
		va[k] = mxtrans(aToB, A.vert(sub + APART_LANES * k < A.nv ? sub + APART_LANES * k : 0));
		vb[k] = B.vert(sub + APART_LANES * k < B.nv ? sub + APART_LANES * k : 0);
	}
	f3 v = aToB.p;
	for (int round = 0; round < APART_ROUNDS; round++)
	{
		const float l2 = dot(v, v);
		if (!(l2 > need * need))
			return false;
		float ha = FLT_BIG, hb = FLT_BIG;
		f3 pa = va[0], pb = vb[0];
#pragma unroll
		for (int k = 0; k < APART_HELD; k++)
		{
			const float h = dot(v, va[k]), g = -dot(v, vb[k]);
			if (h < ha) { ha = h; pa = va[k]; }
			if (g < hb) { hb = g; pb = vb[k]; }
		}
		for (int i = sub + APART_LANES * APART_HELD; i < A.nv; i += APART_LANES)
		{
			const f3 p = mxtrans(aToB, A.vert(i));
			const float h = dot(v, p);
			if (h < ha) { ha = h; pa = p; }
		}
		for (int i = sub + APART_LANES * APART_HELD; i < B.nv; i += APART_LANES)
		{
			const f3 p = B.vert(i);
			const float h = -dot(v, p);
			if (h < hb) { hb = h; pb = p; }
		}
		groupMin(ha, pa);
		groupMin(hb, pb);
		const float g = ha + hb;
		if (g > 0.0f && g * g > need * need * l2)
			return true;
		if (!(l2 - g > 1e-3f * l2))
			return false;   // v is nearest: the gap is |v|
		const f3 d = pa - pb - v;
		const float t = -dot(v, d) / dot(d, d);
		v = v + d * fminf(fmaxf(t, 0.0f), 1.0f);
	}
	return false;
}

// The edges of each polytope whose bounding sphere comes within lim of the
// other polytope's bounding box (both in B's frame, from the staged vertices),
// listed in index order in L.elA / L.elB; every edge when lim is FLT_BIG.
PXH_D void nearEdges(const Poly& A, const Poly& B, CvxLds& L, int lane, float lim, int& nA, int& nB)
{
	const float BIG = FLT_BIG;
	f3 aMin = mk(BIG, BIG, BIG), aMax = -aMin, bMin = aMin, bMax = aMax;
	if (lane < A.nv)
	{
		aMin = ldsV(L.va, lane);
		aMax = aMin;
	}
	if (lane < B.nv)
	{
		bMin = ldsV(L.vb, lane);
		bMax = bMin;
	}
	for (int off = 32; off >= 1; off >>= 1)
	{
		aMin = mk(fminf(aMin.x, __shfl_xor(aMin.x, off)), fminf(aMin.y, __shfl_xor(aMin.y, off)),
		          fminf(aMin.z, __shfl_xor(aMin.z, off)));
		aMax = mk(fmaxf(aMax.x, __shfl_xor(aMax.x, off)), fmaxf(aMax.y, __shfl_xor(aMax.y, off)),
		          fmaxf(aMax.z, __shfl_xor(aMax.z, off)));
		bMin = mk(fminf(bMin.x, __shfl_xor(bMin.x, off)), fminf(bMin.y, __shfl_xor(bMin.y, off)),
		          fminf(bMin.z, __shfl_xor(bMin.z, off)));
		bMax = mk(fmaxf(bMax.x, __shfl_xor(bMax.x, off)), fmaxf(bMax.y, __shfl_xor(bMax.y, off)),
		          fmaxf(bMax.z, __shfl_xor(bMax.z, off)));
	}
	nA = 0;
	nB = 0;
	for (int side = 0; side < 2; side++)
	{
		const int ne = side ? B.ne : A.ne;
		const f3 lo = side ? aMin : bMin, hi = side ? aMax : bMax;
		int cnt = 0;
		for (int base = 0; base < ne; base += 64)
		{
			const int e = base + lane;
			bool keep = false;
			if (e < ne)
			{
				const uint32_t g = side ? L.eb[e] : L.ea[e];
				const float4* vv = side ? L.vb : L.va;
				const f3 p0 = ldsV(vv, int(g & 0xFF)), p1 = ldsV(vv, int((g >> 8) & 0xFF));
				const f3 mid = (p0 + p1) * 0.5f, h = (p1 - p0) * 0.5f;
				const f3 q = mk(fminf(fmaxf(mid.x, lo.x), hi.x), fminf(fmaxf(mid.y, lo.y), hi.y),
				                fminf(fmaxf(mid.z, lo.z), hi.z));
				const f3 dq = mid - q;
				keep = !(sqrtf(dot(dq, dq)) - sqrtf(dot(h, h)) > lim);
			}
			const uint64_t m = __ballot(keep);
			if (keep)
			{
				const int at = cnt + int(__popcll(m & ((1ull << lane) - 1ull)));
				(side ? L.elB : L.elA)[at] = uint8_t(e);
			}
			cnt += int(__popcll(m));
		}
		(side ? nB : nA) = cnt;
	}
	waveSync();
}

// The face axes of polySeparation over the wave, from the staged vertices and
// planes only: B's (order 0 | f << 8 | vertex), then A's (order 1 | ...). The
// lane's least penetrating axis goes to best, bi and its most separating one
// to gap, gi (kind << 24 | f); sep is set on every lane when some axis shows no
// penetration. True when some axis separates the polytopes by more than cd.
PXH_D bool faceAxesWave(const Poly& A, const Poly& B, float cd, const CvxLds& L, int lane, float& best, uint32_t& bi,
                        bool& sep, float& gap, uint32_t& gi)
{
	const float BIG = FLT_BIG;
	best = BIG;
	bi = 0xFFFFFFFFu;
	gap = 0.0f;
	gi = 0;
	bool far = false;
	sep = false;
	for (int f = lane; f < B.np; f += 64)
	{
		const float4 pl = L.pb[f];
		float mn = BIG;
		int vi = 0;
		for (int i = 0; i < A.nv; i++)
		{
			const float4 v = L.va[i];
			const float h = pl.x * v.x + pl.y * v.y + pl.z * v.z + pl.w;
			if (h < mn) { mn = h; vi = i; }
		}
		far |= mn > cd;
		sep |= mn > 0.0f;
		if (mn > gap)
		{
			gap = mn;
			gi = uint32_t(f);
		}
		if (!(mn > 0.0f) && -mn < best)
		{
			best = -mn;
			bi = (uint32_t(f) << 8) | uint32_t(vi);
		}
	}
	for (int f = lane; f < A.np; f += 64)
	{
		const float4 pl = L.pa[f];
		float mn = BIG;
		int vi = 0;
		for (int i = 0; i < B.nv; i++)
		{
			const float4 v = L.vb[i];
			const float h = pl.x * v.x + pl.y * v.y + pl.z * v.z + pl.w;
			if (h < mn) { mn = h; vi = i; }
		}
		far |= mn > cd;
		sep |= mn > 0.0f;
		if (mn > gap)
		{
			gap = mn;
			gi = (1u << 24) | uint32_t(f);
		}
		if (!(mn > 0.0f) && -mn < best)
		{
			best = -mn;
			bi = (1u << 24) | (uint32_t(f) << 8) | uint32_t(vi);
		}
	}
	sep = waveAny(sep);
	return waveAny(far);
}

// The axis of edge pair k (ea * CVX_WAVE_E + eb), whose arcs cross: its overlap
// goes to best, bi if it is smaller, or equal and the pair comes first
PXH_D void edgeAxis(const CvxLds& L, int k, f3 bmean, float& best, uint32_t& bi, bool& sep)
{
	const int ea = k / CVX_WAVE_E, ebi = k - ea * CVX_WAVE_E;
	const uint32_t e = L.ea[ea], g = L.eb[ebi];
	const f3 a0 = ldsV(L.va, int(e & 0xFF)), a1 = ldsV(L.va, int((e >> 8) & 0xFF));
	const f3 b0 = ldsV(L.vb, int(g & 0xFF)), b1 = ldsV(L.vb, int((g >> 8) & 0xFF));
	f3 ax = cross(a1 - a0, b1 - b0);
	const float l2 = dot(ax, ax);
	if (l2 < 1e-12f)
		return;
	ax = ax * (1.0f / sqrtf(l2));
	if (dot(ax, b0 - bmean) < 0.0f)
		ax = -ax;
	const float ov = dot(ax, b0) - dot(ax, a0);
	const uint32_t code = (2u << 24) | uint32_t(k);
	if (ov < 0.0f)
		sep = true;
	else if (ov < best || (ov == best && code < bi))
	{
		best = ov;
		bi = code;
	}
}

PXH_D float edgePairSq(const CvxLds& L, int ea, int eb, f3& c1, f3& c2)
{
	const uint32_t e = L.ea[ea], g = L.eb[eb];
	return segClosestSq(ldsV(L.va, int(e & 0xFF)), ldsV(L.va, int((e >> 8) & 0xFF)), ldsV(L.vb, int(g & 0xFF)),
	                    ldsV(L.vb, int((g >> 8) & 0xFF)), c1, c2);
}

// The entries i < n of the wave with keep(i), listed in index order
template <class K> PXH_D int waveList(int n, int lane, uint8_t* out, K keep)
{
	int cnt = 0;
	for (int base = 0; base < n; base += 64)
	{
		const int i = base + lane;
		const bool k = i < n && keep(i);
		const uint64_t m = __ballot(k);
		if (k)
			out[cnt + int(__popcll(m & ((1ull << lane) - 1ull)))] = uint8_t(i);
		cnt += int(__popcll(m));
	}
	return cnt;
}

PXH_D float waveMin(float v)
{
	for (int off = 32; off >= 1; off >>= 1)
		v = fminf(v, __shfl_xor(v, off));
	return v;
}

// The rest of polySeparation over the wave (same results), after
// faceAxesWave found no axis farther than cd; A, B in LDS as staged
PXH_D void polySeparationWave(const Poly& A, const mxf& aToB, const Poly& B, CvxLds& L, int lane, float best,
                              uint32_t bi, bool sep, float gap, uint32_t gi, float& dist, f3& n, f3& cA, f3& cB)
{
	const float BIG = FLT_BIG;
	const bool slab = sep;   // some face axis separates
	if (!sep)
	{
		f3 bmean = mk(0.0f, 0.0f, 0.0f);
		for (int i = 0; i < B.nv; i++)
			bmean = bmean + ldsV(L.vb, i);
		bmean = bmean * (1.0f / float(B.nv));
		// Edge pairs: each lane holds one of A's edges (its Gauss-map arc in
		// registers) and walks the arcs of B's edges, laid out CVX_ARCS at a time
		// and read as LDS broadcasts. A block of R < 64 of A's edges gives each
		// edge S = 64 / R lanes, which split B's edges between them. Few pairs'
		// arcs cross (about one in 50 for hulls of 24 points), but one or two of
		// every 64 do, and their axis costs three times the arc test: the crossing
		// pairs are listed and measured 64 at a time.
		int cnt = 0;
		for (int b0 = 0; b0 < B.ne; b0 += CVX_ARCS)
		{
			const int nb0 = min(CVX_ARCS, B.ne - b0);
			if (lane < nb0)
			{
				const uint32_t g = L.eb[b0 + lane];
				const f3 nc = -ldsV(L.pb, int((g >> 16) & 0xFF)), nd = -ldsV(L.pb, int(g >> 24));
				const f3 dxc = cross(nd, nc);
				L.arc[3 * lane] = f4(nc, dxc.x);
				L.arc[3 * lane + 1] = f4(nd, dxc.y);
				L.arc[3 * lane + 2].x = dxc.z;
			}
			waveSync();
			for (int base = 0; base < A.ne; base += 64)
			{
				const int R = min(64, A.ne - base), S = 64 / R, part = lane / R;
				const bool has = part < S;
				const int ea = base + (has ? lane - part * R : 0);
				const uint32_t e = L.ea[ea];
				const f3 na = ldsV(L.pa, int((e >> 16) & 0xFF)), nb = ldsV(L.pa, int(e >> 24));
				const f3 bxa = cross(nb, na);
				for (int i0 = 0; i0 < nb0; i0 += S)
				{
					const int i = i0 + part;
					bool arcs = has && i < nb0;
					const int at = arcs ? 3 * i : 0;
					const float4 c = L.arc[at], d = L.arc[at + 1];
					const f3 nc = mk(c), nd = mk(d), dxc = mk(c.w, d.w, L.arc[at + 2].x);
					const float cba = dot(nc, bxa), dba = dot(nd, bxa), adc = dot(na, dxc), bdc = dot(nb, dxc);
					arcs = arcs && cba * dba < 0.0f && adc * bdc < 0.0f && cba * bdc > 0.0f;
					const uint64_t m = __ballot(arcs);
					if (m == 0ull)
						continue;
					if (arcs)
						L.open[cnt + int(__popcll(m & ((1ull << lane) - 1ull)))] = uint32_t(ea * CVX_WAVE_E + b0 + i);
					cnt += int(__popcll(m));
					if (cnt >= 64)
					{
						cnt -= 64;
						waveSync();
						edgeAxis(L, int(L.open[cnt + lane]), bmean, best, bi, sep);
						waveSync();
					}
				}
			}
			waveSync();
		}
		if (lane < cnt)
			edgeAxis(L, int(L.open[lane]), bmean, best, bi, sep);
		sep = waveAny(sep);
		waveSync();
	}
	if (!sep)
	{
		waveArgMin(best, bi);
		if (bi == 0xFFFFFFFFu)
		{
			dist = FLT_BIG;
			return;
		}
		const uint32_t kind = bi >> 24;
		if (kind == 2u)
		{
			const int k = int(bi & 0xFFFFFFu), ea = k / CVX_WAVE_E, ebi = k - ea * CVX_WAVE_E;
			const uint32_t e = L.ea[ea], g = L.eb[ebi];
			const f3 a0 = ldsV(L.va, int(e & 0xFF)), a1 = ldsV(L.va, int((e >> 8) & 0xFF));
			const f3 b0 = ldsV(L.vb, int(g & 0xFF)), b1 = ldsV(L.vb, int((g >> 8) & 0xFF));
			f3 bmean = mk(0.0f, 0.0f, 0.0f);
			for (int i = 0; i < B.nv; i++)
				bmean = bmean + ldsV(L.vb, i);
			bmean = bmean * (1.0f / float(B.nv));
			f3 ax = cross(a1 - a0, b1 - b0);
			ax = ax * (1.0f / sqrtf(dot(ax, ax)));
			if (dot(ax, b0 - bmean) < 0.0f)
				ax = -ax;
			f3 c1, c2;
			segClosestSq(a0, a1, b0, b1, c1, c2);
			n = ax;
			cA = c1;
			cB = c2;
		}
		else
		{
			const int f = int((bi >> 8) & 0xFFFFu), vi = int(bi & 0xFFu);
			if (kind == 0u)
			{
				const float4 pl = L.pb[f];
				const f3 bn = mk(pl.x, pl.y, pl.z), va = ldsV(L.va, vi);
				const float mn = dot(bn, va) + pl.w;
				n = bn;
				cA = va;
				cB = va - bn * mn;
			}
			else
			{
				const float4 pl = L.pa[f];
				const f3 an = mk(pl.x, pl.y, pl.z), vb = ldsV(L.vb, vi);
				const float mn = dot(an, vb) + pl.w;
				n = -an;
				cB = vb;
				cA = vb - an * mn;
			}
		}
		dist = -best;
		return;
	}
	// Separated: closest features (B faces x A vertices, A faces x B vertices,
	// edge pairs), the first minimum in that order.
	//
	// The edges that meet at the closest two vertices hold a pair at squared
	// distance U, so the minimum is no larger. Along the face axis that
	// separates the polytopes most, A's heights less B's bound every distance
	// from below: a vertex or an edge whose height alone is farther from the
	// other polytope than lim = sqrt(U) plus a margin holds no closest feature. The
	// margin is above what planes lie off their polygons' vertices and well above
	// rounding: a height or a distance is off by a few units in the last place (6e-8
	// each) of the largest coordinate, the margin is 1e-5 of what bounds that.
	// What is left keeps its order and its indices, so the first minimum is unchanged.
	int nA, nB;
	float minA = 0.0f, maxB = 0.0f;
	if (slab)
	{
		float g = -gap;
		waveArgMin(g, gi);
		const bool onA = (gi >> 24) != 0u;
		const float4 pl = (onA ? L.pa : L.pb)[gi & 0xFFFFu];
		const f3 sn = onA ? -mk(pl) : mk(pl);
		const float sd = onA ? -pl.w : pl.w;
		float ha = BIG, hb = -BIG;
		if (lane < A.nv)
			L.va[lane].w = ha = dot(sn, ldsV(L.va, lane)) + sd;
		if (lane < B.nv)
			L.vb[lane].w = hb = dot(sn, ldsV(L.vb, lane)) + sd;
		minA = waveMin(ha);
		maxB = -waveMin(-hb);
	}
	float near = BIG;
	uint32_t ni = 0;
	FlatPair fv(lane, B.nv);
	for (int k = lane; k < A.nv * B.nv; k += 64, fv.next())
	{
		const f3 w = ldsV(L.va, fv.i) - ldsV(L.vb, fv.j);
		const float s = dot(w, w);
		if (s < near)
		{
			near = s;
			ni = uint32_t(fv.i << 8 | fv.j);
		}
	}
	waveArgMin(near, ni);
	const uint32_t ia = ni >> 8, ib = ni & 0xFFu;
	nA = waveList(A.ne, lane, L.elA, [&](int e) { return (L.ea[e] & 0xFF) == ia || ((L.ea[e] >> 8) & 0xFF) == ia; });
	nB = waveList(B.ne, lane, L.elB, [&](int e) { return (L.eb[e] & 0xFF) == ib || ((L.eb[e] >> 8) & 0xFF) == ib; });
	waveSync();
	float U = BIG;
	FlatPair fu(lane, nB);
	for (int k = lane; k < nA * nB; k += 64, fu.next())
	{
		f3 c1, c2;
		U = fminf(U, edgePairSq(L, L.elA[fu.i], L.elB[fu.j], c1, c2));
	}
	U = waveMin(U);
	const float extent = fabsf(aToB.p.x) + fabsf(aToB.p.y) + fabsf(aToB.p.z) + A.radius + B.radius;
	const float margin = 1e-4f + 1e-5f * extent + A.slack + B.slack;
	float lim = U < BIG ? sqrtf(U) + margin : BIG;
	waveSync();
	float d2 = BIG;
	uint32_t di = 0xFFFFFFFFu;
	nA = waveList(A.nv, lane, L.elA, [&](int i) { return !(slab && L.va[i].w - maxB > lim); });
	nB = waveList(B.nv, lane, L.elB, [&](int i) { return !(slab && minA - L.vb[i].w > lim); });
	waveSync();
	FlatPair fb(lane, nA);
	for (int k = lane; k < B.np * nA; k += 64, fb.next())
	{
		const int f = fb.i, i = L.elA[fb.j];
		const float4 pl = L.pb[f];
		const f3 bn = mk(pl), va = ldsV(L.va, i);
		const float h = dot(bn, va) + pl.w;
		if (h < 0.0f || h * h >= d2 || h * h > U)
			continue;
		if (!inPolygon(B, f, va - bn * h))
			continue;
		d2 = h * h;
		di = uint32_t(f * A.nv + i);
	}
	FlatPair fa(lane, nB);
	for (int k = lane; k < A.np * nB; k += 64, fa.next())
	{
		const int f = fa.i, i = L.elB[fa.j];
		const float4 pl = L.pa[f];
		const f3 an = mk(pl), vb = ldsV(L.vb, i);
		const float h = dot(an, vb) + pl.w;
		if (h < 0.0f || h * h >= d2 || h * h > U)
			continue;
		if (!inPolygon(A, f, mxtransinv(aToB, vb - an * h)))
			continue;
		d2 = h * h;
		di = (1u << 24) | uint32_t(f * B.nv + i);
	}
	U = waveMin(fminf(U, d2));
	lim = U < BIG ? sqrtf(U) + margin : BIG;
	waveSync();
	if (slab)
	{
		nA = waveList(A.ne, lane, L.elA, [&](int e) {
			return !(fminf(L.va[L.ea[e] & 0xFF].w, L.va[(L.ea[e] >> 8) & 0xFF].w) - maxB > lim);
		});
		nB = waveList(B.ne, lane, L.elB, [&](int e) {
			return !(minA - fmaxf(L.vb[L.eb[e] & 0xFF].w, L.vb[(L.eb[e] >> 8) & 0xFF].w) > lim);
		});
		waveSync();
	}
	else
		nearEdges(A, B, L, lane, lim, nA, nB);
	FlatPair fe(lane, nB);
	for (int k = lane; k < nA * nB; k += 64, fe.next())
	{
		const int ea = L.elA[fe.i], ebi = L.elB[fe.j];
		f3 c1, c2;
		const float s = edgePairSq(L, ea, ebi, c1, c2);
		if (s < d2)
		{
			d2 = s;
			di = (2u << 24) | uint32_t(ea * B.ne + ebi);
		}
	}
	waveArgMin(d2, di);
	if (di == 0xFFFFFFFFu)
	{
		dist = FLT_BIG;   // no feature pair (an empty polytope)
		return;
	}
	const uint32_t kind = di >> 24, k = di & 0xFFFFFFu;
	if (kind == 0u)
	{
		const int f = int(k) / A.nv, i = int(k) - f * A.nv;
		const float4 pl = L.pb[f];
		const f3 bn = mk(pl.x, pl.y, pl.z), va = ldsV(L.va, i);
		cA = va;
		cB = va - bn * (dot(bn, va) + pl.w);
	}
	else if (kind == 1u)
	{
		const int f = int(k) / B.nv, i = int(k) - f * B.nv;
		const float4 pl = L.pa[f];
		const f3 an = mk(pl.x, pl.y, pl.z), vb = ldsV(L.vb, i);
		cB = vb;
		cA = vb - an * (dot(an, vb) + pl.w);
	}
	else
	{
		const int ea = int(k) / B.ne, ebi = int(k) - ea * B.ne;
		edgePairSq(L, ea, ebi, cA, cB);
	}
	dist = sqrtf(d2);
	n = (cA - cB) * (1.0f / dist);
}

// polySeparation of a box- or convex-convex pair over the wave: dist and n
// (sep = dist, n xyz) and the witnesses cA, cB in B's frame, the same on every lane
PXH_D void convexSeparationWave(const Poly& A, const xf& x0, const Poly& B, const xf& x1, float cd, CvxLds& L,
                                int lane, float4& sep, f3& wA, f3& wB)
{
	const mxf aToB = mxfOf(xinvmul(x1, x0));
	for (int i = lane; i < A.nv; i += 64)
		L.va[i] = f4(mxtrans(aToB, A.vert(i)), 0.0f);
	for (int i = lane; i < B.nv; i += 64)
		L.vb[i] = f4(B.vert(i), 0.0f);
	for (int f = lane; f < A.np; f += 64)
	{
		const f3 an = mmul(aToB.r, A.pn(f));
		L.pa[f] = f4(an, A.pd(f) - dot(an, aToB.p));
	}
	for (int f = lane; f < B.np; f += 64)
		L.pb[f] = f4(B.pn(f), B.pd(f));
	waveSync();
	float best;
	uint32_t bi;
	bool sepd;
	float gap;
	uint32_t gi;
	if (faceAxesWave(A, B, cd, L, lane, best, bi, sepd, gap, gi))
	{
		// farther apart than the contact distance
		sep = make_float4(2.0f * cd + 1.0f, 1.0f, 0.0f, 0.0f);
		wA = wB = mk(0.0f, 0.0f, 0.0f);
		waveSync();
		return;
	}
	// The edges in LDS for both searches, and for separated polytopes (the
	// polygon tests of the closest-feature search) the polygon and vertex-ref
	// arrays too, read through the same accessors; pairs rejected by a face
	// axis above need neither, overlapping ones no polygons. A's vertices and
	// planes in its own frame stay in global memory (cached): keeping them
	// out of LDS lets four waves share a SIMD.
	for (int e = lane; e < A.ne; e += 64)
		L.ea[e] = A.edge(e);
	for (int e = lane; e < B.ne; e += 64)
		L.eb[e] = B.edge(e);
	Poly Al = A, Bl = B;
	if (!A.box)
	{
		if (sepd)
		{
			for (int f = lane; f < A.np; f += 64)
				L.polyA[f] = A.poly[f];
			for (int k = lane; k < 2 * A.ne; k += 64)
				L.vrA[k] = A.vr[k];
			Al.poly = L.polyA; Al.vr = L.vrA;
		}
		Al.ed = L.ea;
	}
	if (sepd)
	{
		for (int f = lane; f < B.np; f += 64)
			L.polyB[f] = B.poly[f];
		for (int k = lane; k < 2 * B.ne; k += 64)
			L.vrB[k] = B.vr[k];
		Bl.poly = L.polyB; Bl.vr = L.vrB;
	}
	Bl.v = L.vb; Bl.pl = L.pb; Bl.ed = L.eb;
	waveSync();
	float dist = 0.0f;
	f3 n = mk(1.0f, 0.0f, 0.0f), cA = mk(0.0f, 0.0f, 0.0f), cB = cA;
	polySeparationWave(Al, aToB, Bl, L, lane, best, bi, sepd, gap, gi, dist, n, cA, cB);
	waveSync();   // the staged data stay in use until every lane is done
	sep.x = dist;
	sep.y = n.x; sep.z = n.y; sep.w = n.z;
	wA = cA;
	wB = cB;
}

// ---------------------------------------------------------------------------
// Contacts of a pair over 16 lanes, or of a hull and a plane over a wave. In one
// lane the polygons, the points and the reduction's candidates lie in scratch
// memory and every face, vertex and edge waits for the one before. Here the lanes
// share the faces, take a vertex or an edge pair each and keep the points in the
// order of the one-lane form, so the choices are the same. 8,192 hulls: pairs 107
// us in lanes, 43 so (90 with a wave each); plane pairs 65 and 20.
// ---------------------------------------------------------------------------
struct ContactLds
{
	float4 p0[HULL_MAX_POLY_VERTS], p1[HULL_MAX_POLY_VERTS];   // the polygons in the reference polygon's frame
	float4 pts[HULL_MAX_CONTACTS];                             // point, separation
};

PXH_D int laneOf(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
PXH_D float laneOf(float v, int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); }
PXH_D f3 laneOf(f3 v, int l) { return mk(laneOf(v.x, l), laneOf(v.y, l), laneOf(v.z, l)); }
PXH_D float4 laneOf(float4 v, int l)
{
	return make_float4(laneOf(v.x, l), laneOf(v.y, l), laneOf(v.z, l), laneOf(v.w, l));
}

PXH_D int laneRank(uint64_t m, int lane) { return int(__popcll(m & ((1ull << lane) - 1ull))); }

// Groups of 16 lanes, as many as a polygon may have vertices: lane i of a group is
// gl = i; the lanes of a group always take the same way
constexpr int GROUP = 16;
static_assert(HULL_MAX_POLY_VERTS <= GROUP, "a polygon's vertices take a lane each");
PXH_D uint32_t groupBallot(bool b) { return uint32_t(__ballot(b) >> (__lane_id() & 48)) & 0xFFFFu; }
PXH_D float groupLane(float v, int i) { return __shfl(v, i, GROUP); }
PXH_D f3 groupLane(f3 v, int i) { return mk(groupLane(v.x, i), groupLane(v.y, i), groupLane(v.z, i)); }
PXH_D int groupRank(uint32_t m, int gl) { return __popc(m & ((1u << gl) - 1u)); }
PXH_D void groupArgMin(float& v, uint32_t& idx)
{
	for (int off = GROUP / 2; off >= 1; off >>= 1)
	{
		const float ov = __shfl_xor(v, off);
		const uint32_t oi = __shfl_xor(idx, off);
		if (ov < v || (ov == v && oi < idx))
		{
			v = ov;
			idx = oi;
		}
	}
}

template <int LANES> PXH_D void lanesArgMin(float& v, uint32_t& idx)
{
	if constexpr (LANES == 64)
		waveArgMin(v, idx);
	else
		groupArgMin(v, idx);
}

// witnessPolygon over LANES lanes (64 or a group)
template <int LANES> PXH_D int witnessPolygonLanes(const Poly& P, f3 normal, f3 closest, float tolerance, int lane)
{
	const float eps = -tolerance;
	float minDist = FLT_BIG, least = FLT_BIG;   // least: minus the largest distance
	uint32_t first = 0u, maxIdx = 0xFFFFFFFFu;
	if (lane > 0)
		first = 0xFFFFFFFFu;
	for (int i = lane; i < P.np; i += LANES)
	{
		const float dist = dot(P.pn(i), closest) + P.pd(i);
		const float pdi = dist >= eps ? fabsf(dist) : FLT_BIG;
		if (minDist > pdi) { minDist = pdi; first = uint32_t(i); }
		if (-dist < least) { least = -dist; maxIdx = uint32_t(i); }
	}
	lanesArgMin<LANES>(minDist, first);
	if (minDist == FLT_BIG)
	{
		lanesArgMin<LANES>(least, maxIdx);
		return maxIdx == 0xFFFFFFFFu ? 0 : int(maxIdx);
	}
	const float firstProj = dot(normalize(P.pn(int(first))), normal);
	float bestProj = firstProj;
	uint32_t idx = 0xFFFFFFFFu;
	for (int i = lane; i < P.np; i += LANES)
	{
		const f3 pn = P.pn(i);
		const float di = dot(pn, closest) + P.pd(i);
		const float pdi = di >= eps ? fabsf(di) : FLT_BIG;
		if ((tolerance > (pdi - minDist)) && (int(first) != i))
		{
			const float proj = dot(normalize(pn), normal);
			if (bestProj > proj) { idx = uint32_t(i); bestProj = proj; }
		}
	}
	lanesArgMin<LANES>(bestProj, idx);
	return idx == 0xFFFFFFFFu ? int(first) : int(idx);
}

// the bounds of a group's points, widened
PXH_D void groupBounds(bool has, f3 p, f3& mn, f3& mx)
{
	const float feps = 1.1920928955078125e-7f;
	mn = has ? p : mk(FLT_BIG, FLT_BIG, FLT_BIG);
	mx = has ? p : -mk(FLT_BIG, FLT_BIG, FLT_BIG);
	for (int off = GROUP / 2; off >= 1; off >>= 1)
	{
		mn.x = fminf(mn.x, __shfl_xor(mn.x, off));
		mn.y = fminf(mn.y, __shfl_xor(mn.y, off));
		mx.x = fmaxf(mx.x, __shfl_xor(mx.x, off));
		mx.y = fmaxf(mx.y, __shfl_xor(mx.y, off));
	}
	mn = mn - mk(feps, feps, feps);
	mx = mx + mk(feps, feps, feps);
}

// generatedContacts (geomutils/src/pcm/GuPCMContactGenBoxConvex.cpp:331-530) into
// L.pts: reference polygon `ref` of P0, incident polygon `inc` of P1, t0To1 maps
// P0's frame to P1's; the points on P1 (its frame, onP1) or on P0's reference
// plane (its frame), first the incident vertices inside, then the reference ones,
// then the edge crossings; their number
PXH_D int generatedContactsGroup(const Poly& P0, const Poly& P1, int ref, int inc, const mxf& t0To1, float cd, bool onP1,
                                ContactLds& L, int gl)
{
	const f3 n = normalize(P0.pn(ref));
	const m33 rot = rotFromZ(n);
	const int nr = P0.pcount(ref), ni = P1.pcount(inc);
	const bool isRef = gl < nr, isInc = gl < ni;
	f3 q0 = mk(0.0f, 0.0f, 0.0f), q1 = q0, vert1 = q0, mn, mx;
	if (isRef)
	{
		q0 = mmul(rot, P0.vert(P0.pvert(ref, gl)));
		L.p0[gl] = f4(q0, 0.0f);
	}
	const float d = groupLane(q0.z, 0), rd = d + cd;
	float t1 = 0.0f;
	bool pen = false;
	if (isInc)
	{
		vert1 = P1.vert(P1.pvert(inc, gl));
		q1 = mmul(rot, mxtransinv(t0To1, vert1));
		const float z = q1.z;
		t1 = z - d;
		q1.z = d;
		L.p1[gl] = f4(q1, t1);
		pen = rd > z;
	}
	const uint32_t pens = groupBallot(pen);
	const f3 sPoint = groupLane(vert1, 0);
	waveSync();
	groupBounds(isRef, q0, mn, mx);
	bool in = pen && polyContainsN(L.p0, nr, q1, mn, mx);
	uint32_t m = groupBallot(in);
	if (in)
		L.pts[groupRank(m, gl)] = f4(onP1 ? vert1 : mtmul(rot, q1), t1);
	int nc = __popc(m);
	if (nc == ni)
		return nc;
	groupBounds(isInc, q1, mn, mx);
	const f3 incN = normalize(P1.pn(inc));
	const f3 nIn1 = mmul(t0To1.r, n);
	in = isRef && polyContainsN(L.p1, ni, q0, mn, mx);
	f3 vert0 = q0, a = q0;
	float t = 0.0f;
	if (in)
	{
		vert0 = mtmul(rot, q0);
		a = mxtrans(t0To1, vert0);
		t = dot(incN, sPoint - a) / dot(incN, nIn1);
		in = !(t > cd);
	}
	m = groupBallot(in);
	if (in)
		L.pts[nc + groupRank(m, gl)] = f4(onP1 ? nIn1 * t + a : vert0, t);
	const int inside = __popc(m);
	nc += inside;
	if (inside == nr)
		return nc;
	for (int k0 = 0; k0 < ni * nr; k0 += GROUP)
	{
		const int k = k0 + gl;
		bool hit = k < ni * nr;
		f3 pt = q0;
		float sep = 0.0f;
		if (hit)
		{
			const int iS = k / nr, rS = k - iS * nr, iE = iS == 0 ? ni - 1 : iS - 1, rE = rS == 0 ? nr - 1 : rS - 1;
			const float4 sA = L.p1[iS], sB = L.p1[iE];
			const f3 ipA = mk(sA), ipB = mk(sB), rpA = mk(L.p0[rS]), rpB = mk(L.p0[rE]);
			const float a1 = triArea2(rpA, rpB, ipA), a2 = triArea2(rpA, rpB, ipB);
			const float a3 = triArea2(ipA, ipB, rpA), a4 = triArea2(ipA, ipB, rpB);
			hit = (((pens >> iS) | (pens >> iE)) & 1u) != 0u &&
			      !(fminf(ipA.x, ipB.x) > fmaxf(rpA.x, rpB.x) || fminf(ipA.y, ipB.y) > fmaxf(rpA.y, rpB.y) ||
			        fminf(rpA.x, rpB.x) > fmaxf(ipA.x, ipB.x) || fminf(rpA.y, rpB.y) > fmaxf(ipA.y, ipB.y)) &&
			      0.0f > a1 * a2 && 0.0f > a3 * a4;
			if (hit)
			{
				const f3 ipAO = mk(ipA.x, ipA.y, sA.w + d), ipBO = mk(ipB.x, ipB.y, sB.w + d);
				const float u = a1 / (a2 - a1);
				const f3 pBB = ipAO - (ipBO - ipAO) * u;
				const f3 pAA = mk(pBB.x, pBB.y, d);
				sep = pBB.z - pAA.z;
				hit = !(sep > cd);
				pt = onP1 ? mxtrans(t0To1, mtmul(rot, pBB)) : mtmul(rot, pAA);
			}
		}
		m = groupBallot(hit);
		const int to = nc + groupRank(m, gl);
		if (hit && to < HULL_MAX_CONTACTS)
			L.pts[to] = f4(pt, sep);
		nc += __popc(m);
		if (nc >= HULL_MAX_CONTACTS)
			return HULL_MAX_CONTACTS;
	}
	return nc;
}

// Reduction to four (PersistentContactManifold::addBatchManifoldContacts,
// geomutils/src/pcm/GuPersistentContactManifold.cpp:805-830, reduceBatchContacts
// :1008-1172) of the group's points in LDS (their common normal cn0): their
// number, and in lane i the i-th. The points are the candidate list: one that is
// taken leaves its place to the last.
PXH_D int batchReduceGroup(float4* pts, int n, f3 cn0, float tol, int gl, float4& out)
{
	out = pts[gl < n ? gl : 0];
	if (n <= 4)
		return n;
	int nc = n;
	auto drop = [&](int ci) {
		nc--;
		const float4 last = pts[nc];
		waveSync();
		if (gl == 0)
			pts[ci] = last;
		waveSync();
	};
	// the first candidate of the least value, -1 if none is below FLT_BIG
	auto least = [&](auto value, float& v) {
		v = FLT_BIG;
		uint32_t idx = 0xFFFFFFFFu;
		for (int i = gl; i < nc; i += GROUP)
		{
			const float x = value(pts[i]);
			if (x < v) { v = x; idx = uint32_t(i); }
		}
		groupArgMin(v, idx);
		return int(idx);
	};
	float maxPen, minPen, maxDist, minDist;
	int ci = max(least([](float4 c) { return c.w; }, maxPen), 0);
	least([](float4 c) { return -c.w; }, minPen);
	minPen = -minPen;
	float4 ch[4];
	ch[0] = pts[ci];
	const f3 b0 = mk(ch[0]);
	drop(ci);
	ci = max(least([&](float4 c) { const f3 v = mk(c) - b0; return -dot(v, v); }, maxDist), 0);
	ch[1] = pts[ci];
	drop(ci);
	f3 nrm = cross(mk(ch[1]) - b0, cn0);
	const float sq = dot(nrm, nrm);
	if (sq > 0.0f) { const float len = sqrtf(sq); nrm = mk(nrm.x / len, nrm.y / len, nrm.z / len); } else nrm = cn0;
	auto height = [&](float4 c) { return dot(mk(c) - b0, nrm); };
	ci = max(least([&](float4 c) { return -height(c); }, maxDist), 0);
	maxDist = -maxDist;
	int ci1 = max(least(height, minDist), 0);
	ch[2] = pts[ci];
	ch[3] = pts[ci1];
	drop(ci);
	if (nc == ci1)
		ci1 = ci;
	if (minDist * maxDist > 0.0f)
	{
		const int far = least([&](float4 c) { return -height(c); }, maxDist);
		if (far >= 0)
		{
			ci1 = far;
			ch[3] = pts[far];
		}
	}
	drop(ci1);
	const float eps = tol * 0.02f;
	if (eps > maxPen && minPen > eps)
	{
#pragma unroll
		for (int i = 0; i < 4; i++)
		{
			const float pen = ch[i].w;
			if (pen > eps)
			{
				float v;
				const int c = least([&](float4 q) { return pen > q.w && eps > q.w ? q.w : FLT_BIG; }, v);
				if (c >= 0)
				{
					const float4 orig = ch[i];
					ch[i] = pts[c];
					waveSync();
					if (gl == 0)
						pts[c] = orig;
					waveSync();
				}
			}
		}
	}
	out = gl == 0 ? ch[0] : gl == 1 ? ch[1] : gl == 2 ? ch[2] : ch[3];
	return 4;
}

// Contacts of a box- or convex-convex pair no farther apart than cd, from its
// separation (dist, n from B towards A, closest points or minimum-translation
// witnesses cA, cB in B's frame), into contact slot `slot`: witness polygons,
// clipping and reduction to four, as Gu::pcmContactConvexConvex /
// pcmContactBoxConvex on a fresh manifold
// (geomutils/src/pcm/GuPCMContactConvexConvex.cpp:111-276, GuPCMContactBoxConvex.cpp;
// Gu::generateFullContactManifold and Gu::addGJKEPAContacts,
// GuPCMContactGenBoxConvex.cpp:532-720); points on shape1 in the world and the
// summed normal (PersistentContactManifold::addManifoldContactsToContactBuffer /
// getWorldNormal, GuPersistentContactManifold.cpp:739-762,
// GuPersistentContactManifold.h:405-416)
PXH_D void convexContactsGroup(const Poly& A, const xf& x0, const Poly& B, const xf& x1, float dist, f3 n, f3 cA, f3 cB,
                              float cd, float tol, ContactLds& L, int gl, int64_t slot, float4* ctN, float4* ctP)
{
	const mxf aToB = mxfOf(xinvmul(x1, x0));
	const float lo = tol * 1e-2f, hi = tol * 5e-2f;
	const float tA = fminf(fmaxf(A.margin, lo), hi), tB = fminf(fmaxf(B.margin, lo), hi);
	const f3 negN = -n;
	const f3 nIn0 = mtmul(aToB.r, n);
	const int f1 = witnessPolygonLanes<GROUP>(B, negN, cB, tB, gl);
	const int f0 = witnessPolygonLanes<GROUP>(A, nIn0, mxtransinv(aToB, cA), tA, gl);
	const f3 refN = normalize(B.pn(f1)), incN = normalize(A.pn(f0));
	f3 ln;
	int nc;
	if (fabsf(dot(refN, negN)) >= fabsf(dot(incN, nIn0)))
	{
		const mxf bToA = mxfOf(xinvmul(x0, x1));
		nc = generatedContactsGroup(B, A, f1, f0, bToA, cd, false, L, gl);
		ln = refN;
	}
	else
	{
		nc = generatedContactsGroup(A, B, f0, f1, aToB, cd, true, L, gl);
		ln = -mmul(aToB.r, incN);
	}
	waveSync();
	float4 pt = f4(cB, dist);
	if (nc == 0)
	{
		// the closest-feature / minimum-translation point stays the only point
		ln = n;
		nc = 1;
	}
	else
		nc = batchReduceGroup(L.pts, nc, ln, tol, gl, pt);
	f3 s = ln;
	for (int i = 1; i < nc; i++)
		s = s + ln;
	const bool keep = gl < nc && cd >= pt.w;
	const uint32_t m = groupBallot(keep);
	if (keep)
		ctP[4 * slot + groupRank(m, gl)] = f4(xtrans(x1, mk(pt)), pt.w);
	if (gl == 0)
		ctN[slot] = f4(normalize(qrot(x1.q, s)), __int_as_float(int(__popc(m))));
	waveSync();
}

// Gu::pcmContactPlaneConvex on a fresh manifold
// (geomutils/src/pcm/GuPCMContactPlaneConvex.cpp:36-227) into contact slot `slot`,
// the normal from the plane to the hull: the face most opposed to the plane
// normal, or the better face of the edge whose summed face normals are most
// opposed to it (5e-4 bias towards edges); the chosen face's vertices below the
// contact distance, taken once more when an edge was chosen (the reference
// passes over the same face twice); reduced to four.
// Deliberate deviation: when the chosen face does not hold the hull's deepest
// vertex (an irregular hull can rest on a vertex that the face most opposed to
// the plane does not contain), that vertex joins the batch. The reference scene's
// persistent manifold keeps such a vertex from earlier steps; a step that
// generates contacts afresh has to add it.
PXH_D void planeConvexWave(f3 pn, float pd, const Poly& B, const xf& tb, float cd, float tol, ContactLds& L, int lane,
                           int64_t slot, float4* ctN, float4* ctP)
{
	const f3 n = normalize(qrotinv(tb.q, pn));
	const f3 nn = -n;
	float minProj = FLT_BIG;
	uint32_t faceIdx = lane == 0 ? 0u : 0xFFFFFFFFu;
	for (int i = lane; i < B.np; i += 64)
	{
		const float proj = dot(n, B.pn(i));
		if (minProj > proj) { minProj = proj; faceIdx = uint32_t(i); }
	}
	waveArgMin(minProj, faceIdx);
	int face = faceIdx == 0xFFFFFFFFu ? 0 : int(faceIdx);
	int edgeSel = -1;
	minProj = minProj - 5e-4f;
	float maxDpSq = minProj * minProj;
	for (int base = 0; base < B.ne; base += 64)
	{
		// the next edge of the block that beats the best so far, until none does
		const bool has = base + lane < B.ne;
		const uint32_t g = B.edge(has ? base + lane : 0);
		const f3 en = B.pn(int((g >> 16) & 0xFF)) + B.pn(int(g >> 24));
		const float enMagSq = dot(en, en);
		const float dp = dot(en, nn);
		const float sqDp = dp * dp;
		int from = 0;
		while (from < 64)
		{
			const uint64_t m = __ballot(has && lane >= from && dp >= 0.0f && sqDp > maxDpSq * enMagSq);
			if (m == 0ull)
				break;
			const int l = __ffsll((unsigned long long)m) - 1;
			maxDpSq = laneOf(sqDp / enMagSq, l);
			edgeSel = base + l;
			from = l + 1;
		}
	}
	int passes = 1;
	if (edgeSel >= 0)
	{
		const uint32_t g = B.edge(edgeSel);
		const int f0 = int((g >> 16) & 0xFF), f1 = int(g >> 24);
		face = dot(B.pn(f0), nn) > dot(B.pn(f1), nn) ? f0 : f1;
		passes = 2;
	}
	float deepest = FLT_BIG;
	uint32_t dv = lane == 0 ? 0u : 0xFFFFFFFFu;
	for (int i = lane; i < B.nv; i += 64)
	{
		const float s = dot(pn, xtrans(tb, B.vert(i))) + pd;
		if (s < deepest) { deepest = s; dv = uint32_t(i); }
	}
	waveArgMin(deepest, dv);
	if (dv == 0xFFFFFFFFu)
		dv = 0u;
	const int cnt = B.pcount(face);
	bool below = lane < passes * cnt, isDeepest = false;
	f3 pw = pn;
	float s = 0.0f;
	if (below)
	{
		const int vi = B.pvert(face, lane < cnt ? lane : lane - cnt);
		pw = xtrans(tb, B.vert(vi));
		s = dot(pn, pw) + pd;
		below = cd > s;
		isDeepest = vi == int(dv);
	}
	const uint64_t m = __ballot(below);
	if (below)
		L.pts[laneRank(m, lane)] = f4(pw - pn * s, s);
	int nc = int(__popcll(m));
	if (!__any(below && isDeepest) && cd > deepest && nc < HULL_MAX_CONTACTS)
	{
		const f3 dw = xtrans(tb, B.vert(int(dv)));
		if (lane == 0)
			L.pts[nc] = f4(dw - pn * deepest, deepest);
		nc++;
	}
	waveSync();
	float4 pt = f4(pn, 0.0f);
	if (nc > 0)
		nc = batchReduceGroup(L.pts, nc, pn, tol, lane & (GROUP - 1), pt);
	const bool keep = lane < nc && cd >= pt.w;
	const uint64_t k = __ballot(keep);
	if (keep)
		ctP[4 * slot + laneRank(k, lane)] = pt;
	if (lane == 0)
		ctN[slot] = f4(pn, __int_as_float(int(__popcll(k))));
	waveSync();
}

}  // namespace pxh
