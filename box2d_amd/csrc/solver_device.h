// SPDX-FileCopyrightText: 2022 Erin Catto (Box2D; the contact solver arithmetic below restates its
// src/contact_solver.c and src/solver.c in the same operation order)
// SPDX-License-Identifier: MIT
// GPU solver arithmetic for one contact or joint constraint.
//
// These functions are the per-lane bodies of the constraint kernels. The colored path reproduces
// the reference's wide (SIMD lane) arithmetic, including its operation order, its a >= b / a <= b
// min-max semantics and the fact that a one-point manifold still runs the second point with zeros
// (reference src/contact_solver.c:936-1063, 1811-2228). The overflow path reproduces the scalar
// overflow solver (src/contact_solver.c:24-545), whose expressions differ from the wide ones.
// Joints are in joints_device.h.
#pragma once

#include "layout.h"

namespace b2g
{

#define B2G_DEVI __device__ __forceinline__

// Float arrays of one allocation, field-major: field k of element i is at base[k * stride + i].
struct FieldTable
{
	float* base;
	int stride;

	__host__ __device__ float* operator[]( int field ) const
	{
		return base + (size_t)field * stride;
	}
};

// One field of a RowTable.
struct RowField
{
	float* p;

	__host__ __device__ float& operator[]( int i ) const
	{
		return p[4 * (size_t)i];
	}
};

// The constraint fields (ConstraintField): one allocation, one float4 array of `stride` constraints
// per group of four fields. A lane loads the groups a stage needs with 7 to 9 16-byte loads instead
// of about 30 4-byte ones. table[k][i] is field k of constraint i; Group( g )[i] is group g's four.
struct RowTable
{
	float* base;
	int stride;

	__host__ __device__ RowField operator[]( int field ) const
	{
		return RowField{ base + 4 * (size_t)( field >> 2 ) * stride + ( field & 3 ) };
	}
	__host__ __device__ float4* Group( int group ) const
	{
		return reinterpret_cast<float4*>( base ) + (size_t)group * stride;
	}
};

struct ConstraintSoA
{
	RowTable f;
	int* bodyA; // body ids (GlobalBodies view)
	int* bodyB;
	int* contactId;
	int* pointCount;
	int* slotA; // LDS slots of the fused solver (LdsBodies, PackedBodies views)
	int* slotB;
};

// LDS body slots of the fused solver: every static body reads the identity state kept in slot 0,
// awake bodies occupy slots 1..count (at most kFusedBodyCapacity).
constexpr int kFusedBodyCapacity = 5400;
constexpr int kStaticSlot = 0;

// Workgroup barrier that orders LDS accesses only: global loads issued before it stay in flight.
B2G_DEVI void LdsBarrier()
{
	__builtin_amdgcn_fence( __ATOMIC_RELEASE, "workgroup", "local" );
	__builtin_amdgcn_s_barrier();
	__builtin_amdgcn_fence( __ATOMIC_ACQUIRE, "workgroup", "local" );
}

B2G_DEVI float MaxW( float a, float b )
{
	return a >= b ? a : b;
}

B2G_DEVI float MinW( float a, float b )
{
	return a <= b ? a : b;
}

B2G_DEVI Softness MakeSoft( float hertz, float zeta, float h )
{
	if ( hertz == 0.0f )
	{
		return Softness{ 0.0f, 0.0f, 0.0f };
	}
	float omega = 2.0f * B2_PI * hertz;
	float a1 = 2.0f * zeta + h * omega;
	float a2 = h * omega * a1;
	float a3 = 1.0f / ( 1.0f + a2 );
	return Softness{ omega / a1, a2 * a3, a3 };
}

// Deterministic arctangent (reference src/math_functions.c:96-136).
B2G_DEVI float Atan2( float y, float x )
{
	if ( x == 0.0f && y == 0.0f )
	{
		return 0.0f;
	}
	float ax = b2AbsFloat( x );
	float ay = b2AbsFloat( y );
	float mx = b2MaxFloat( ay, ax );
	float mn = b2MinFloat( ay, ax );
	float a = mn / mx;
	float s = a * a;
	float c = s * a;
	float q = s * s;
	float r = 0.024840285f * q + 0.18681418f;
	float t = -0.094097948f * q - 0.33213072f;
	r = r * s + t;
	r = r * c + a;
	if ( ay > ax )
	{
		r = 1.57079637f - r;
	}
	if ( x < 0 )
	{
		r = 3.14159274f - r;
	}
	if ( y < 0 )
	{
		r = -r;
	}
	return r;
}

struct LaneBody
{
	float vx, vy, w;
	uint32_t flags;
	float dpx, dpy, dqc, dqs;
};

// Body state access of the solver functions. GlobalBodies reads and writes the id-indexed state
// array in device memory; LdsBodies reads and writes a world's awake bodies staged in LDS by
// solver-set index (the fused solver kernel). Constraint and joint body indices must match the
// view: body ids for GlobalBodies, LDS slots for LdsBodies.
struct GlobalBodies
{
	BodyState* states;

	B2G_DEVI LaneBody Load( int index ) const
	{
		const float4* p = reinterpret_cast<const float4*>( states + index );
		float4 a = p[0];
		float4 b = p[1];
		LaneBody r;
		r.vx = a.x;
		r.vy = a.y;
		r.w = a.z;
		r.flags = __float_as_uint( a.w );
		r.dpx = b.x;
		r.dpy = b.y;
		r.dqc = b.z;
		r.dqs = b.w;
		return r;
	}

	// Delta position and rotation only (the fields no solver stage writes).
	B2G_DEVI void LoadDelta( int index, b2Vec2& dp, b2Rot& dq ) const
	{
		float4 b = reinterpret_cast<const float4*>( states + index )[1];
		dp = { b.x, b.y };
		dq = { b.z, b.w };
	}

	// Velocities are written back for dynamic bodies only (kinematic and static states are read-only).
	B2G_DEVI void Store( int index, const LaneBody& b ) const
	{
		if ( b.flags & kDynamicFlag )
		{
			BodyState* s = states + index;
			s->linearVelocity.x = b.vx;
			s->linearVelocity.y = b.vy;
			s->angularVelocity = b.w;
		}
	}

	static constexpr bool kJointBodiesLoaded = true; // JointA, JointB come from the joint's record
	B2G_DEVI static int JointA( const JointSim* j )
	{
		return j->indexA;
	}
	B2G_DEVI static int JointB( const JointSim* j )
	{
		return j->indexB;
	}
};

struct LdsBodies
{
	float* vx;
	float* vy;
	float* w;
	float* dpx;
	float* dpy;
	float* dqc;
	float* dqs;
	uint16_t* flags;

	B2G_DEVI LaneBody Load( int index ) const
	{
		LaneBody r;
		r.vx = vx[index];
		r.vy = vy[index];
		r.w = w[index];
		r.flags = flags[index];
		r.dpx = dpx[index];
		r.dpy = dpy[index];
		r.dqc = dqc[index];
		r.dqs = dqs[index];
		return r;
	}

	B2G_DEVI void LoadDelta( int index, b2Vec2& dp, b2Rot& dq ) const
	{
		dp = { dpx[index], dpy[index] };
		dq = { dqc[index], dqs[index] };
	}

	B2G_DEVI void Store( int index, const LaneBody& b ) const
	{
		if ( b.flags & kDynamicFlag )
		{
			vx[index] = b.vx;
			vy[index] = b.vy;
			w[index] = b.w;
		}
	}

	static constexpr bool kJointBodiesLoaded = true; // JointA, JointB come from the joint's record
	B2G_DEVI static int JointA( const JointSim* j )
	{
		return j->slotA;
	}
	B2G_DEVI static int JointB( const JointSim* j )
	{
		return j->slotB;
	}
};

// A world's awake bodies in LDS as the fused solver keeps them: the delta pose as one 16-byte word,
// the velocity as three floats (12 bytes, so that neighbouring slots fall into different banks) and
// the flags, 30 bytes per slot.
struct PackedBodies
{
	float4* d;
	float* v;
	uint16_t* flags;

	B2G_DEVI LaneBody Load( int index ) const
	{
		float4 p = d[index];
		LaneBody r;
		r.vx = v[3 * index];
		r.vy = v[3 * index + 1];
		r.w = v[3 * index + 2];
		r.flags = flags[index];
		r.dpx = p.x;
		r.dpy = p.y;
		r.dqc = p.z;
		r.dqs = p.w;
		return r;
	}

	B2G_DEVI void LoadDelta( int index, b2Vec2& dp, b2Rot& dq ) const
	{
		float4 p = d[index];
		dp = { p.x, p.y };
		dq = { p.z, p.w };
	}

	B2G_DEVI void StoreVelocity( int index, float vx, float vy, float w ) const
	{
		v[3 * index] = vx;
		v[3 * index + 1] = vy;
		v[3 * index + 2] = w;
	}

	B2G_DEVI void Store( int index, const LaneBody& b ) const
	{
		if ( b.flags & kDynamicFlag )
		{
			StoreVelocity( index, b.vx, b.vy, b.w );
		}
	}

	static constexpr bool kJointBodiesLoaded = true; // JointA, JointB come from the joint's record
	B2G_DEVI static int JointA( const JointSim* j )
	{
		return j->slotA;
	}
	B2G_DEVI static int JointB( const JointSim* j )
	{
		return j->slotB;
	}
};

// ---------------------------------------------------------------------------------------------
// Body integration

// What velocity integration adds and multiplies, the same in every substep of a step.
struct VelocityStep
{
	b2Vec2 linearVelocityDelta;
	float linearDamping;
	float angularVelocityDelta;
	float angularDamping;
};

B2G_DEVI VelocityStep MakeVelocityStep( const BodySim& sim, const StepParams& p )
{
	float h = p.h;
	VelocityStep s;
	s.linearDamping = 1.0f / ( 1.0f + h * sim.linearDamping );
	s.angularDamping = 1.0f / ( 1.0f + h * sim.angularDamping );
	float gravityScale = sim.invMass > 0.0f ? sim.gravityScale : 0.0f;
	s.linearVelocityDelta = b2Add( b2MulSV( h * sim.invMass, sim.force ), b2MulSV( h * gravityScale, p.gravity ) );
	s.angularVelocityDelta = h * sim.invInertia * sim.torque;
	return s;
}

// Velocity integration of one body (reference src/solver.c:66-112).
B2G_DEVI void ApplyVelocityStep( const VelocityStep& s, b2Vec2& v, float& w )
{
	v = b2MulAdd( s.linearVelocityDelta, s.linearDamping, v );
	w = s.angularVelocityDelta + s.angularDamping * w;
}

B2G_DEVI void IntegrateVelocity( const BodySim& sim, BodyState* state, const StepParams& p )
{
	ApplyVelocityStep( MakeVelocityStep( sim, p ), state->linearVelocity, state->angularVelocity );
}

// Position integration of one body: locks, speed caps, delta position and rotation
// (reference src/solver.c:114-162).
B2G_DEVI void IntegratePosition( BodyState* state, const StepParams& p )
{
	float h = p.h;
	float maxLinearSpeed = p.maxLinearVelocity;
	float maxAngularSpeed = ( 0.25f * B2_PI ) * p.inv_dt;
	float maxLinearSpeedSquared = maxLinearSpeed * maxLinearSpeed;
	float maxAngularSpeedSquared = maxAngularSpeed * maxAngularSpeed;

	b2Vec2 v = state->linearVelocity;
	float w = state->angularVelocity;
	uint32_t flags = state->flags;

	v.x = ( flags & kLockLinearX ) ? 0.0f : v.x;
	v.y = ( flags & kLockLinearY ) ? 0.0f : v.y;
	w = ( flags & kLockAngularZ ) ? 0.0f : w;

	if ( b2Dot( v, v ) > maxLinearSpeedSquared )
	{
		float ratio = maxLinearSpeed / b2Length( v );
		v = b2MulSV( ratio, v );
		flags |= kIsSpeedCapped;
	}

	if ( w * w > maxAngularSpeedSquared && ( flags & kAllowFastRotation ) == 0 )
	{
		float ratio = maxAngularSpeed / b2AbsFloat( w );
		w *= ratio;
		flags |= kIsSpeedCapped;
	}

	state->flags = flags;
	state->linearVelocity = v;
	state->angularVelocity = w;
	state->deltaPosition = b2MulAdd( state->deltaPosition, h, v );
	state->deltaRotation = b2IntegrateRotation( state->deltaRotation, h * w );
}

// ---------------------------------------------------------------------------------------------
// Colored (wide-lane) contact arithmetic
//
// A lane holds its constraint as a ContactRow (the groups its stage loaded) and the velocities of
// its two bodies; the impulse groups i1, i2 (normal, tangent, total normal impulse) and the rolling
// impulse are updated in the row and stored by the caller.

struct ContactRow
{
	float4 mass;	// invMassA, invIA, invMassB, invIB
	float4 normal;	// x, y, friction, tangent speed
	float4 soft;	// bias rate, mass scale, impulse scale, restitution
	float4 rolling; // resistance, mass, impulse
	float4 a1, m1, i1;
	float4 a2, m2, i2;
};

enum RowGroup
{
	kgMass = kcInvMassA / 4,
	kgNormal = kcNormalX / 4,
	kgSoft = kcBiasRate / 4,
	kgRolling = kcRollingResistance / 4,
	kgAnchor1 = kcAnchorA1X / 4,
	kgPoint1 = kcBaseSeparation1 / 4,
	kgImpulse1 = kcNormalImpulse1 / 4,
	kgAnchor2 = kcAnchorA2X / 4,
	kgPoint2 = kcBaseSeparation2 / 4,
	kgImpulse2 = kcNormalImpulse2 / 4,
};

enum ColorStage
{
	kStageWarmStart,
	kStageSolve,
	kStageRelax,
	kStageRestitution,
};

// The groups a stage reads (the others stay as they are).
template <int Stage>
B2G_DEVI void LoadRow( const ConstraintSoA& c, int i, ContactRow& r )
{
	r.mass = c.f.Group( kgMass )[i];
	r.normal = c.f.Group( kgNormal )[i];
	if ( Stage == kStageSolve )
	{
		r.soft = c.f.Group( kgSoft )[i];
	}
	else
	{
		r.rolling = c.f.Group( kgRolling )[i];
	}
	r.a1 = c.f.Group( kgAnchor1 )[i];
	r.i1 = c.f.Group( kgImpulse1 )[i];
	r.a2 = c.f.Group( kgAnchor2 )[i];
	r.i2 = c.f.Group( kgImpulse2 )[i];
	if ( Stage != kStageWarmStart )
	{
		r.m1 = c.f.Group( kgPoint1 )[i];
		r.m2 = c.f.Group( kgPoint2 )[i];
	}
}

B2G_DEVI void StoreRowImpulses( const ConstraintSoA& c, int i, const ContactRow& r )
{
	c.f.Group( kgImpulse1 )[i] = r.i1;
	c.f.Group( kgImpulse2 )[i] = r.i2;
}

struct PairVel
{
	float vAx, vAy, wA, vBx, vBy, wB;
};

// Velocity change of an impulse (Px, Py) at a point with anchors a.
B2G_DEVI void ApplyRowImpulse( PairVel& v, const ContactRow& r, const float4& a, float Px, float Py )
{
	v.vAx = v.vAx - r.mass.x * Px;
	v.vAy = v.vAy - r.mass.x * Py;
	v.wA = v.wA - r.mass.y * ( a.x * Py - a.y * Px );
	v.vBx = v.vBx + r.mass.z * Px;
	v.vBy = v.vBy + r.mass.z * Py;
	v.wB = v.wB + r.mass.w * ( a.z * Py - a.w * Px );
}

B2G_DEVI void WarmStartRowPoint( PairVel& v, const ContactRow& r, const float4& a, float4& imp )
{
	float nX = r.normal.x, nY = r.normal.y;
	float tX = nY;
	float tY = 0.0f - nX;
	float Px = imp.x * nX + imp.y * tX;
	float Py = imp.x * nY + imp.y * tY;
	v.wA = v.wA - r.mass.y * ( a.x * Py - a.y * Px );
	v.vAx = v.vAx - r.mass.x * Px;
	v.vAy = v.vAy - r.mass.x * Py;
	v.wB = v.wB + r.mass.w * ( a.z * Py - a.w * Px );
	v.vBx = v.vBx + r.mass.z * Px;
	v.vBy = v.vBy + r.mass.z * Py;
	imp.z = imp.z + imp.x;
}

B2G_DEVI void WarmStartRow( ContactRow& r, PairVel& v )
{
	WarmStartRowPoint( v, r, r.a1, r.i1 );
	WarmStartRowPoint( v, r, r.a2, r.i2 );
	v.wA = v.wA - r.mass.y * r.rolling.z;
	v.wB = v.wB + r.mass.w * r.rolling.z;
}

// The part of a normal point's solve that depends on the delta poses only, which no stage changes
// between two position integrations.
struct PointBias
{
	float bias, massScale, impulseScale;
};

struct RowBias
{
	PointBias p1, p2;
};

template <bool kUseBias>
B2G_DEVI PointBias RowPointBias( const ContactRow& r, const float4& a, const float4& m, float dpX, float dpY, const float4& dA,
								 const float4& dB, float inv_h, float contactSpeed )
{
	// moving anchors for the current separation
	float rsAx = dA.z * a.x - dA.w * a.y;
	float rsAy = dA.w * a.x + dA.z * a.y;
	float rsBx = dB.z * a.z - dB.w * a.w;
	float rsBy = dB.w * a.z + dB.z * a.w;

	float dsx = dpX + ( rsBx - rsAx );
	float dsy = dpY + ( rsBy - rsAy );
	float s = ( r.normal.x * dsx + r.normal.y * dsy ) + m.x;

	float biasRate = kUseBias ? r.soft.y * r.soft.x : 0.0f;
	float massScale = kUseBias ? r.soft.y : 1.0f;
	float impulseScale = kUseBias ? r.soft.z : 0.0f;

	bool mask = s > 0.0f;
	float specBias = s * inv_h;
	float softBias = MaxW( biasRate * s, contactSpeed );
	PointBias out;
	out.bias = mask ? specBias : softBias;
	out.massScale = mask ? 1.0f : massScale;
	out.impulseScale = mask ? 0.0f : impulseScale;
	return out;
}

// dA, dB: delta position (x, y) and rotation (c, s) of the two bodies.
template <bool kUseBias>
B2G_DEVI RowBias ComputeRowBias( const ContactRow& r, const float4& dA, const float4& dB, float inv_h, float contactSpeed )
{
	float dpX = dB.x - dA.x;
	float dpY = dB.y - dA.y;
	RowBias b;
	b.p1 = RowPointBias<kUseBias>( r, r.a1, r.m1, dpX, dpY, dA, dB, inv_h, contactSpeed );
	b.p2 = RowPointBias<kUseBias>( r, r.a2, r.m2, dpX, dpY, dA, dB, inv_h, contactSpeed );
	return b;
}

B2G_DEVI void SolveRowNormal( PairVel& v, const ContactRow& r, const float4& a, const float4& m, float4& imp, const PointBias& b )
{
	float nX = r.normal.x, nY = r.normal.y;
	float dvx = ( v.vBx - v.wB * a.w ) - ( v.vAx - v.wA * a.y );
	float dvy = ( v.vBy + v.wB * a.z ) - ( v.vAy + v.wA * a.x );
	float vn = dvx * nX + dvy * nY;

	float negImpulse = m.y * ( b.massScale * vn + b.bias ) + b.impulseScale * imp.x;
	float newImpulse = MaxW( imp.x - negImpulse, 0.0f );
	float impulse = newImpulse - imp.x;
	imp.x = newImpulse;
	imp.z = imp.z + impulse;
	ApplyRowImpulse( v, r, a, impulse * nX, impulse * nY );
}

B2G_DEVI void SolveRowFriction( PairVel& v, const ContactRow& r, const float4& a, const float4& m, float4& imp )
{
	float tX = r.normal.y;
	float tY = 0.0f - r.normal.x;
	float dvx = ( v.vBx - v.wB * a.w ) - ( v.vAx - v.wA * a.y );
	float dvy = ( v.vBy + v.wB * a.z ) - ( v.vAy + v.wA * a.x );
	float vt = dvx * tX + dvy * tY;
	vt = vt - r.normal.w;

	float negImpulse = m.z * vt;
	float maxFriction = r.normal.z * imp.x;
	float newImpulse = imp.y - negImpulse;
	newImpulse = MaxW( 0.0f - maxFriction, MinW( newImpulse, maxFriction ) );
	float impulse = newImpulse - imp.y;
	imp.y = newImpulse;
	ApplyRowImpulse( v, r, a, impulse * tX, impulse * tY );
}

// The velocity part of the solve (kUseBias) or relax stage. laneGroupRolling: any constraint of this
// constraint's 4-lane group has rolling resistance (the wide solver tests the whole group).
template <bool kUseBias>
B2G_DEVI void SolveRow( ContactRow& r, PairVel& v, const RowBias& b, bool laneGroupRolling )
{
	float totalNormalImpulse = 0.0f;
	SolveRowNormal( v, r, r.a1, r.m1, r.i1, b.p1 );
	totalNormalImpulse = totalNormalImpulse + r.i1.x;
	SolveRowNormal( v, r, r.a2, r.m2, r.i2, b.p2 );
	totalNormalImpulse = totalNormalImpulse + r.i2.x;

	if ( kUseBias == false )
	{
		if ( laneGroupRolling )
		{
			float deltaLambda = r.rolling.y * ( v.wA - v.wB );
			float lambda = r.rolling.z;
			float maxLambda = r.rolling.x * totalNormalImpulse;
			float rolling = b2ClampFloat( lambda + deltaLambda, -maxLambda, maxLambda );
			r.rolling.z = rolling;
			deltaLambda = rolling - lambda;
			v.wA = v.wA - r.mass.y * deltaLambda;
			v.wB = v.wB + r.mass.w * deltaLambda;
		}
		SolveRowFriction( v, r, r.a1, r.m1, r.i1 );
		SolveRowFriction( v, r, r.a2, r.m2, r.i2 );
	}
}

B2G_DEVI PairVel ToPair( const LaneBody& bA, const LaneBody& bB )
{
	return PairVel{ bA.vx, bA.vy, bA.w, bB.vx, bB.vy, bB.w };
}

template <typename Bodies>
B2G_DEVI void StorePair( const Bodies& B, int ia, int ib, LaneBody& bA, LaneBody& bB, const PairVel& v )
{
	bA.vx = v.vAx;
	bA.vy = v.vAy;
	bA.w = v.wA;
	bB.vx = v.vBx;
	bB.vy = v.vBy;
	bB.w = v.wB;
	B.Store( ia, bA );
	B.Store( ib, bB );
}

template <typename Bodies>
B2G_DEVI void WarmStartContact( const ConstraintSoA& c, int i, const Bodies& B )
{
	int ia = c.bodyA[i];
	int ib = c.bodyB[i];
	ContactRow r;
	LoadRow<kStageWarmStart>( c, i, r );
	LaneBody bA = B.Load( ia );
	LaneBody bB = B.Load( ib );
	PairVel v = ToPair( bA, bB );
	WarmStartRow( r, v );
	StoreRowImpulses( c, i, r );
	StorePair( B, ia, ib, bA, bB, v );
}

// rolling( row ): whether the constraint's 4-lane group has rolling resistance (relax stage only).
template <bool kUseBias, typename Bodies, typename Rolling>
B2G_DEVI void SolveContact( const ConstraintSoA& c, int i, const Bodies& B, float inv_h, float contactSpeed, Rolling rolling )
{
	int ia = c.bodyA[i];
	int ib = c.bodyB[i];
	ContactRow r;
	LoadRow<kUseBias ? kStageSolve : kStageRelax>( c, i, r );
	LaneBody bA = B.Load( ia );
	LaneBody bB = B.Load( ib );
	float4 dA = make_float4( bA.dpx, bA.dpy, bA.dqc, bA.dqs );
	float4 dB = make_float4( bB.dpx, bB.dpy, bB.dqc, bB.dqs );
	RowBias bias = ComputeRowBias<kUseBias>( r, dA, dB, inv_h, contactSpeed );
	PairVel v = ToPair( bA, bB );
	bool laneGroupRolling = kUseBias == false && rolling( r );
	SolveRow<kUseBias>( r, v, bias, laneGroupRolling );
	StoreRowImpulses( c, i, r );
	if ( laneGroupRolling )
	{
		c.f[kcRollingImpulse][i] = r.rolling.z;
	}
	StorePair( B, ia, ib, bA, bB, v );
}

// ---------------------------------------------------------------------------------------------
// The same arithmetic with two neighbouring lanes per constraint, the even one for body A and the odd
// one for body B: each holds its own body's velocity, anchors and masses. The terms of the relative
// velocity are formed in both lanes at once and exchanged within the pair, and each lane applies the
// impulse to its own body, which takes a quarter of the instructions off a constraint's serial path
// and halves its LDS traffic. Body A's masses are negated: v - m * P and v + ( -m ) * P are the same
// float, so every value is that of the one-lane form.

// x of the pair's lane A and of its lane B (DPP quad permutations).
B2G_DEVI float PairA( float x )
{
	return __uint_as_float( __builtin_amdgcn_mov_dpp( __float_as_uint( x ), 0xA0, 0xF, 0xF, true ) ); // 0, 0, 2, 2
}

B2G_DEVI float PairB( float x )
{
	return __uint_as_float( __builtin_amdgcn_mov_dpp( __float_as_uint( x ), 0xF5, 0xF, 0xF, true ) ); // 1, 1, 3, 3
}

// Native vectors: a row in flight is one register tuple per load.
typedef float F2 __attribute__( ( ext_vector_type( 2 ) ) );
typedef float F4 __attribute__( ( ext_vector_type( 4 ) ) );

B2G_DEVI F4 PairGroup( const ConstraintSoA& c, int group, int i )
{
	return reinterpret_cast<const F4*>( c.f.Group( group ) )[i];
}

struct PairRow
{
	F2 mass;	// own inverse mass and inertia, negated for body A
	F4 normal;	// x, y, friction, tangent speed
	F4 soft;	// bias rate, mass scale, impulse scale, -
	F4 rolling; // resistance, mass, impulse, -
	F2 a1, a2;	// own anchors
	F4 m1, m2;	// base separation, normal mass, tangent mass, -
	F4 i1, i2;	// normal, tangent, total normal impulse, -
};

// The groups a stage reads (the others stay as they are).
template <int Stage>
B2G_DEVI void LoadPairRow( const ConstraintSoA& c, int i, int side, PairRow& r )
{
	r.mass = reinterpret_cast<const F2*>( c.f.Group( kgMass ) + i )[side];
	r.normal = PairGroup( c, kgNormal, i );
	if ( Stage == kStageSolve )
	{
		r.soft = PairGroup( c, kgSoft, i );
	}
	else
	{
		r.rolling = PairGroup( c, kgRolling, i );
	}
	r.a1 = reinterpret_cast<const F2*>( c.f.Group( kgAnchor1 ) + i )[side];
	r.i1 = PairGroup( c, kgImpulse1, i );
	r.a2 = reinterpret_cast<const F2*>( c.f.Group( kgAnchor2 ) + i )[side];
	r.i2 = PairGroup( c, kgImpulse2, i );
	if ( Stage != kStageWarmStart )
	{
		r.m1 = PairGroup( c, kgPoint1, i );
		r.m2 = PairGroup( c, kgPoint2, i );
	}
}

// Lane A stores point 1's impulses, lane B point 2's.
B2G_DEVI void StorePairImpulses( const ConstraintSoA& c, int i, int side, const PairRow& r )
{
	F4 impulse;
	impulse.x = side == 0 ? r.i1.x : r.i2.x;
	impulse.y = side == 0 ? r.i1.y : r.i2.y;
	impulse.z = side == 0 ? r.i1.z : r.i2.z;
	impulse.w = 0.0f;
	reinterpret_cast<F4*>( c.f.Group( side == 0 ? kgImpulse1 : kgImpulse2 ) )[i] = impulse;
}

struct OwnVel
{
	float x, y, w;
};

B2G_DEVI void ApplyPairImpulse( OwnVel& v, F2 mass, F2 a, float Px, float Py )
{
	v.x = v.x + mass.x * Px;
	v.y = v.y + mass.x * Py;
	v.w = v.w + mass.y * ( a.x * Py - a.y * Px );
}

B2G_DEVI void WarmStartPairPoint( OwnVel& v, const PairRow& r, F2 mass, F2 a, F4& imp )
{
	float nX = r.normal.x, nY = r.normal.y;
	float tX = nY;
	float tY = 0.0f - nX;
	float Px = imp.x * nX + imp.y * tX;
	float Py = imp.x * nY + imp.y * tY;
	ApplyPairImpulse( v, mass, a, Px, Py );
	imp.z = imp.z + imp.x;
}

B2G_DEVI void WarmStartPair( PairRow& r, F2 mass, OwnVel& v )
{
	WarmStartPairPoint( v, r, mass, r.a1, r.i1 );
	WarmStartPairPoint( v, r, mass, r.a2, r.i2 );
	v.w = v.w + mass.y * r.rolling.z;
}

// d: own delta position (x, y) and rotation (c, s).
template <bool kUseBias>
B2G_DEVI PointBias PairPointBias( const PairRow& r, F2 a, const F4& m, float dpX, float dpY, const F4& d, float inv_h,
								  float contactSpeed )
{
	float rsx = d.z * a.x - d.w * a.y;
	float rsy = d.w * a.x + d.z * a.y;
	float dsx = dpX + ( PairB( rsx ) - PairA( rsx ) );
	float dsy = dpY + ( PairB( rsy ) - PairA( rsy ) );
	float s = ( r.normal.x * dsx + r.normal.y * dsy ) + m.x;

	float biasRate = kUseBias ? r.soft.y * r.soft.x : 0.0f;
	bool mask = s > 0.0f;
	float specBias = s * inv_h;
	float softBias = MaxW( biasRate * s, contactSpeed );
	PointBias out;
	out.bias = mask ? specBias : softBias;
	out.massScale = kUseBias == false || mask ? 1.0f : r.soft.y;
	out.impulseScale = kUseBias == false || mask ? 0.0f : r.soft.z;
	return out;
}

template <bool kUseBias>
B2G_DEVI RowBias ComputePairBias( const PairRow& r, const F4& d, float inv_h, float contactSpeed )
{
	float dpX = PairB( d.x ) - PairA( d.x );
	float dpY = PairB( d.y ) - PairA( d.y );
	RowBias b;
	b.p1 = PairPointBias<kUseBias>( r, r.a1, r.m1, dpX, dpY, d, inv_h, contactSpeed );
	b.p2 = PairPointBias<kUseBias>( r, r.a2, r.m2, dpX, dpY, d, inv_h, contactSpeed );
	return b;
}

// Relative velocity of the two bodies at a point along (x, y).
B2G_DEVI float PairRelativeVelocity( const OwnVel& v, F2 a, float x, float y )
{
	float px = v.x - v.w * a.y;
	float py = v.y + v.w * a.x;
	float dvx = PairB( px ) - PairA( px );
	float dvy = PairB( py ) - PairA( py );
	return dvx * x + dvy * y;
}

template <bool kUseBias>
B2G_DEVI void SolvePairNormal( OwnVel& v, const PairRow& r, F2 mass, F2 a, const F4& m, F4& imp, const PointBias& b )
{
	float nX = r.normal.x, nY = r.normal.y;
	float vn = PairRelativeVelocity( v, a, nX, nY );
	// without the bias the scales are 1 and 0 (impulses are finite, so 0 * impulse adds +0)
	float negImpulse = m.y * ( b.massScale * vn + b.bias ) + b.impulseScale * imp.x;
	float newImpulse = MaxW( imp.x - negImpulse, 0.0f );
	float impulse = newImpulse - imp.x;
	imp.x = newImpulse;
	imp.z = imp.z + impulse;
	ApplyPairImpulse( v, mass, a, impulse * nX, impulse * nY );
}

B2G_DEVI void SolvePairFriction( OwnVel& v, const PairRow& r, F2 mass, F2 a, const F4& m, F4& imp )
{
	float tX = r.normal.y;
	float tY = 0.0f - r.normal.x;
	float vt = PairRelativeVelocity( v, a, tX, tY );
	vt = vt - r.normal.w;

	float negImpulse = m.z * vt;
	float maxFriction = r.normal.z * imp.x;
	float newImpulse = imp.y - negImpulse;
	newImpulse = MaxW( 0.0f - maxFriction, MinW( newImpulse, maxFriction ) );
	float impulse = newImpulse - imp.y;
	imp.y = newImpulse;
	ApplyPairImpulse( v, mass, a, impulse * tX, impulse * tY );
}

template <bool kUseBias>
B2G_DEVI void SolvePair( PairRow& r, F2 mass, OwnVel& v, const RowBias& b, bool laneGroupRolling )
{
	float totalNormalImpulse = 0.0f;
	SolvePairNormal<kUseBias>( v, r, mass, r.a1, r.m1, r.i1, b.p1 );
	totalNormalImpulse = totalNormalImpulse + r.i1.x;
	SolvePairNormal<kUseBias>( v, r, mass, r.a2, r.m2, r.i2, b.p2 );
	totalNormalImpulse = totalNormalImpulse + r.i2.x;

	if ( kUseBias == false )
	{
		if ( laneGroupRolling )
		{
			float deltaLambda = r.rolling.y * ( PairA( v.w ) - PairB( v.w ) );
			float lambda = r.rolling.z;
			float maxLambda = r.rolling.x * totalNormalImpulse;
			float rolling = b2ClampFloat( lambda + deltaLambda, -maxLambda, maxLambda );
			r.rolling.z = rolling;
			deltaLambda = rolling - lambda;
			v.w = v.w + mass.y * deltaLambda;
		}
		SolvePairFriction( v, r, mass, r.a1, r.m1, r.i1 );
		SolvePairFriction( v, r, mass, r.a2, r.m2, r.i2 );
	}
}

B2G_DEVI void RestitutionPoint( const ConstraintSoA& c, int i, LaneBody& bA, LaneBody& bB, float mA, float mB, float iA,
								float iB, float nX, float nY, float threshold, float restitution, bool restitutionMask,
								int fAx, int fAy, int fBx, int fBy, int fRelVel, int fTotal, int fNormalMass,
								int fNormalImpulse )
{
	float relativeVelocity = c.f[fRelVel][i];
	bool mask1 = ( relativeVelocity + threshold ) > 0.0f;
	bool mask2 = c.f[fTotal][i] == 0.0f;
	bool mask = mask1 || mask2 || restitutionMask;
	float mass = mask ? 0.0f : c.f[fNormalMass][i];

	float rAx = c.f[fAx][i], rAy = c.f[fAy][i];
	float rBx = c.f[fBx][i], rBy = c.f[fBy][i];

	float dvx = ( bB.vx - bB.w * rBy ) - ( bA.vx - bA.w * rAy );
	float dvy = ( bB.vy + bB.w * rBx ) - ( bA.vy + bA.w * rAx );
	float vn = dvx * nX + dvy * nY;

	float negImpulse = mass * ( vn + restitution * relativeVelocity );
	float normalImpulse = c.f[fNormalImpulse][i];
	float newImpulse = MaxW( normalImpulse - negImpulse, 0.0f );
	float deltaImpulse = newImpulse - normalImpulse;
	c.f[fNormalImpulse][i] = newImpulse;
	c.f[fTotal][i] = c.f[fTotal][i] + deltaImpulse;

	float Px = deltaImpulse * nX;
	float Py = deltaImpulse * nY;
	bA.vx = bA.vx - mA * Px;
	bA.vy = bA.vy - mA * Py;
	bA.w = bA.w - iA * ( rAx * Py - rAy * Px );
	bB.vx = bB.vx + mB * Px;
	bB.vy = bB.vy + mB * Py;
	bB.w = bB.w + iB * ( rBx * Py - rBy * Px );
}

template <typename Bodies>
B2G_DEVI void RestitutionContact( const ConstraintSoA& c, int i, const Bodies& B, float threshold )
{
	int ia = c.bodyA[i];
	int ib = c.bodyB[i];
	LaneBody bA = B.Load( ia );
	LaneBody bB = B.Load( ib );

	float mA = c.f[kcInvMassA][i], mB = c.f[kcInvMassB][i];
	float iA = c.f[kcInvIA][i], iB = c.f[kcInvIB][i];
	float nX = c.f[kcNormalX][i], nY = c.f[kcNormalY][i];
	float restitution = c.f[kcRestitution][i];
	bool restitutionMask = restitution == 0.0f;

	RestitutionPoint( c, i, bA, bB, mA, mB, iA, iB, nX, nY, threshold, restitution, restitutionMask, kcAnchorA1X, kcAnchorA1Y,
					  kcAnchorB1X, kcAnchorB1Y, kcRelativeVelocity1, kcTotalNormalImpulse1, kcNormalMass1, kcNormalImpulse1 );
	RestitutionPoint( c, i, bA, bB, mA, mB, iA, iB, nX, nY, threshold, restitution, restitutionMask, kcAnchorA2X, kcAnchorA2Y,
					  kcAnchorB2X, kcAnchorB2Y, kcRelativeVelocity2, kcTotalNormalImpulse2, kcNormalMass2, kcNormalImpulse2 );

	B.Store( ia, bA );
	B.Store( ib, bB );
}

// ---------------------------------------------------------------------------------------------
// Overflow (scalar) contact arithmetic, solved one constraint after another by a single lane.

B2G_DEVI BodyState ToState( const LaneBody& b )
{
	BodyState s;
	s.linearVelocity = { b.vx, b.vy };
	s.angularVelocity = b.w;
	s.flags = b.flags;
	s.deltaPosition = { b.dpx, b.dpy };
	s.deltaRotation = { b.dqc, b.dqs };
	return s;
}

B2G_DEVI LaneBody ToLane( const BodyState& s )
{
	LaneBody b;
	b.vx = s.linearVelocity.x;
	b.vy = s.linearVelocity.y;
	b.w = s.angularVelocity;
	b.flags = s.flags;
	b.dpx = s.deltaPosition.x;
	b.dpy = s.deltaPosition.y;
	b.dqc = s.deltaRotation.c;
	b.dqs = s.deltaRotation.s;
	return b;
}

struct OverflowVel
{
	float vx, vy, w;
};

template <typename Bodies>
B2G_DEVI void OverflowWarmStart( const ConstraintSoA& c, int i, const Bodies& B )
{
	int ia = c.bodyA[i];
	int ib = c.bodyB[i];
	BodyState sA = ToState( B.Load( ia ) );
	BodyState* stateA = &sA;
	BodyState sB = ToState( B.Load( ib ) );
	BodyState* stateB = &sB;

	b2Vec2 vA = stateA->linearVelocity;
	float wA = stateA->angularVelocity;
	b2Vec2 vB = stateB->linearVelocity;
	float wB = stateB->angularVelocity;

	float mA = c.f[kcInvMassA][i], mB = c.f[kcInvMassB][i];
	float iA = c.f[kcInvIA][i], iB = c.f[kcInvIB][i];
	b2Vec2 normal = { c.f[kcNormalX][i], c.f[kcNormalY][i] };
	b2Vec2 tangent = b2RightPerp( normal );
	int pointCount = c.pointCount[i];

	for ( int j = 0; j < pointCount; ++j )
	{
		int o = j == 0 ? 0 : ( kcAnchorA2X - kcAnchorA1X );
		b2Vec2 rA = { c.f[kcAnchorA1X + o][i], c.f[kcAnchorA1Y + o][i] };
		b2Vec2 rB = { c.f[kcAnchorB1X + o][i], c.f[kcAnchorB1Y + o][i] };
		float ni = c.f[kcNormalImpulse1 + o][i];
		float ti = c.f[kcTangentImpulse1 + o][i];
		b2Vec2 P = b2Add( b2MulSV( ni, normal ), b2MulSV( ti, tangent ) );
		c.f[kcTotalNormalImpulse1 + o][i] = c.f[kcTotalNormalImpulse1 + o][i] + ni;
		wA -= iA * b2Cross( rA, P );
		vA = b2MulAdd( vA, -mA, P );
		wB += iB * b2Cross( rB, P );
		vB = b2MulAdd( vB, mB, P );
	}

	float rolling = c.f[kcRollingImpulse][i];
	wA -= iA * rolling;
	wB += iB * rolling;

	if ( stateA->flags & kDynamicFlag )
	{
		stateA->linearVelocity = vA;
		stateA->angularVelocity = wA;
	}
	if ( stateB->flags & kDynamicFlag )
	{
		stateB->linearVelocity = vB;
		stateB->angularVelocity = wB;
	}

	B.Store( ia, ToLane( sA ) );
	B.Store( ib, ToLane( sB ) );
}

template <typename Bodies>
B2G_DEVI void OverflowSolve( const ConstraintSoA& c, int i, const Bodies& B, bool useBias, float inv_h, float contactSpeed )
{
	float mA = c.f[kcInvMassA][i], mB = c.f[kcInvMassB][i];
	float iA = c.f[kcInvIA][i], iB = c.f[kcInvIB][i];

	int ia = c.bodyA[i];
	int ib = c.bodyB[i];
	BodyState sA = ToState( B.Load( ia ) );
	BodyState* stateA = &sA;
	BodyState sB = ToState( B.Load( ib ) );
	BodyState* stateB = &sB;

	b2Vec2 vA = stateA->linearVelocity;
	float wA = stateA->angularVelocity;
	b2Rot dqA = stateA->deltaRotation;
	b2Vec2 vB = stateB->linearVelocity;
	float wB = stateB->angularVelocity;
	b2Rot dqB = stateB->deltaRotation;

	b2Vec2 dp = b2Sub( stateB->deltaPosition, stateA->deltaPosition );

	b2Vec2 normal = { c.f[kcNormalX][i], c.f[kcNormalY][i] };
	b2Vec2 tangent = b2RightPerp( normal );
	float friction = c.f[kcFriction][i];
	Softness softness = { c.f[kcBiasRate][i], c.f[kcMassScale][i], c.f[kcImpulseScale][i] };
	int pointCount = c.pointCount[i];
	float totalNormalImpulse = 0.0f;

	for ( int j = 0; j < pointCount; ++j )
	{
		int o = j == 0 ? 0 : ( kcAnchorA2X - kcAnchorA1X );
		b2Vec2 rA = { c.f[kcAnchorA1X + o][i], c.f[kcAnchorA1Y + o][i] };
		b2Vec2 rB = { c.f[kcAnchorB1X + o][i], c.f[kcAnchorB1Y + o][i] };

		b2Vec2 ds = b2Add( dp, b2Sub( b2RotateVector( dqB, rB ), b2RotateVector( dqA, rA ) ) );
		float s = c.f[kcBaseSeparation1 + o][i] + b2Dot( ds, normal );

		float velocityBias = 0.0f;
		float massScale = 1.0f;
		float impulseScale = 0.0f;
		if ( s > 0.0f )
		{
			velocityBias = s * inv_h;
		}
		else if ( useBias )
		{
			velocityBias = b2MaxFloat( softness.massScale * softness.biasRate * s, -contactSpeed );
			massScale = softness.massScale;
			impulseScale = softness.impulseScale;
		}

		b2Vec2 vrA = b2Add( vA, b2CrossSV( wA, rA ) );
		b2Vec2 vrB = b2Add( vB, b2CrossSV( wB, rB ) );
		float vn = b2Dot( b2Sub( vrB, vrA ), normal );

		float normalImpulse = c.f[kcNormalImpulse1 + o][i];
		float impulse = -c.f[kcNormalMass1 + o][i] * ( massScale * vn + velocityBias ) - impulseScale * normalImpulse;
		float newImpulse = b2MaxFloat( normalImpulse + impulse, 0.0f );
		impulse = newImpulse - normalImpulse;
		c.f[kcNormalImpulse1 + o][i] = newImpulse;
		c.f[kcTotalNormalImpulse1 + o][i] = c.f[kcTotalNormalImpulse1 + o][i] + impulse;
		totalNormalImpulse += newImpulse;

		b2Vec2 P = b2MulSV( impulse, normal );
		vA = b2MulSub( vA, mA, P );
		wA -= iA * b2Cross( rA, P );
		vB = b2MulAdd( vB, mB, P );
		wB += iB * b2Cross( rB, P );
	}

	if ( useBias == false )
	{
		float tangentSpeed = c.f[kcTangentSpeed][i];
		for ( int j = 0; j < pointCount; ++j )
		{
			int o = j == 0 ? 0 : ( kcAnchorA2X - kcAnchorA1X );
			b2Vec2 rA = { c.f[kcAnchorA1X + o][i], c.f[kcAnchorA1Y + o][i] };
			b2Vec2 rB = { c.f[kcAnchorB1X + o][i], c.f[kcAnchorB1Y + o][i] };

			b2Vec2 vrB = b2Add( vB, b2CrossSV( wB, rB ) );
			b2Vec2 vrA = b2Add( vA, b2CrossSV( wA, rA ) );
			float vt = b2Dot( b2Sub( vrB, vrA ), tangent ) - tangentSpeed;
			float impulse = c.f[kcTangentMass1 + o][i] * ( -vt );
			float maxFriction = friction * c.f[kcNormalImpulse1 + o][i];
			float tangentImpulse = c.f[kcTangentImpulse1 + o][i];
			float newImpulse = b2ClampFloat( tangentImpulse + impulse, -maxFriction, maxFriction );
			impulse = newImpulse - tangentImpulse;
			c.f[kcTangentImpulse1 + o][i] = newImpulse;

			b2Vec2 P = b2MulSV( impulse, tangent );
			vA = b2MulSub( vA, mA, P );
			wA -= iA * b2Cross( rA, P );
			vB = b2MulAdd( vB, mB, P );
			wB += iB * b2Cross( rB, P );
		}

		{
			float deltaLambda = -c.f[kcRollingMass][i] * ( wB - wA );
			float lambda = c.f[kcRollingImpulse][i];
			float maxLambda = c.f[kcRollingResistance][i] * totalNormalImpulse;
			float rolling = b2ClampFloat( lambda + deltaLambda, -maxLambda, maxLambda );
			c.f[kcRollingImpulse][i] = rolling;
			deltaLambda = rolling - lambda;
			wA -= iA * deltaLambda;
			wB += iB * deltaLambda;
		}
	}

	if ( stateA->flags & kDynamicFlag )
	{
		stateA->linearVelocity = vA;
		stateA->angularVelocity = wA;
	}
	if ( stateB->flags & kDynamicFlag )
	{
		stateB->linearVelocity = vB;
		stateB->angularVelocity = wB;
	}

	B.Store( ia, ToLane( sA ) );
	B.Store( ib, ToLane( sB ) );
}

template <typename Bodies>
B2G_DEVI void OverflowRestitution( const ConstraintSoA& c, int i, const Bodies& B, float threshold )
{
	float restitution = c.f[kcRestitution][i];
	if ( restitution == 0.0f )
	{
		return;
	}

	float mA = c.f[kcInvMassA][i], mB = c.f[kcInvMassB][i];
	float iA = c.f[kcInvIA][i], iB = c.f[kcInvIB][i];
	int ia = c.bodyA[i];
	int ib = c.bodyB[i];
	BodyState sA = ToState( B.Load( ia ) );
	BodyState* stateA = &sA;
	BodyState sB = ToState( B.Load( ib ) );
	BodyState* stateB = &sB;
	b2Vec2 vA = stateA->linearVelocity;
	float wA = stateA->angularVelocity;
	b2Vec2 vB = stateB->linearVelocity;
	float wB = stateB->angularVelocity;
	b2Vec2 normal = { c.f[kcNormalX][i], c.f[kcNormalY][i] };
	int pointCount = c.pointCount[i];

	for ( int j = 0; j < pointCount; ++j )
	{
		int o = j == 0 ? 0 : ( kcAnchorA2X - kcAnchorA1X );
		float relativeVelocity = c.f[kcRelativeVelocity1 + o][i];
		if ( relativeVelocity > -threshold || c.f[kcTotalNormalImpulse1 + o][i] == 0.0f )
		{
			continue;
		}

		b2Vec2 rA = { c.f[kcAnchorA1X + o][i], c.f[kcAnchorA1Y + o][i] };
		b2Vec2 rB = { c.f[kcAnchorB1X + o][i], c.f[kcAnchorB1Y + o][i] };
		b2Vec2 vrB = b2Add( vB, b2CrossSV( wB, rB ) );
		b2Vec2 vrA = b2Add( vA, b2CrossSV( wA, rA ) );
		float vn = b2Dot( b2Sub( vrB, vrA ), normal );

		float normalImpulse = c.f[kcNormalImpulse1 + o][i];
		float impulse = -c.f[kcNormalMass1 + o][i] * ( vn + restitution * relativeVelocity );
		float newImpulse = b2MaxFloat( normalImpulse + impulse, 0.0f );
		impulse = newImpulse - normalImpulse;
		c.f[kcNormalImpulse1 + o][i] = newImpulse;
		c.f[kcTotalNormalImpulse1 + o][i] = c.f[kcTotalNormalImpulse1 + o][i] + impulse;

		b2Vec2 P = b2MulSV( impulse, normal );
		vA = b2MulSub( vA, mA, P );
		wA -= iA * b2Cross( rA, P );
		vB = b2MulAdd( vB, mB, P );
		wB += iB * b2Cross( rB, P );
	}

	if ( stateA->flags & kDynamicFlag )
	{
		stateA->linearVelocity = vA;
		stateA->angularVelocity = wA;
	}
	if ( stateB->flags & kDynamicFlag )
	{
		stateB->linearVelocity = vB;
		stateB->angularVelocity = wB;
	}

	B.Store( ia, ToLane( sA ) );
	B.Store( ib, ToLane( sB ) );
}

} // namespace b2g

#include "joints_device.h"

namespace b2g
{

// ---------------------------------------------------------------------------------------------
// Warm start by body

// The warm-start stage of one dynamic body: the velocity deltas of its constraints' accumulated
// impulses applied in the stage's order (overflow joints, overflow contacts, then per color its
// joints and contacts). The deltas depend on impulses, anchors, normals, masses and the body's
// delta rotation, never on velocities, so the per-body sequence of float operations is exactly the
// one the color-by-color stage applies to this body (WarmStartContact, OverflowWarmStart,
// WarmStartJoint). Entries: index << 3 | owner << 2 | joint << 1 | side; the owner entry of a
// contact also accumulates the contact's total normal impulses.
template <typename Bodies>
B2G_DEVI void WarmStartJointSide( const JointSim* joint, bool sideB, const Bodies& B, b2Rot dq, b2Vec2 dp, float& vx, float& vy,
								  float& w )
{
	b2Vec2 dpOther;
	b2Rot dqOther;
	B.LoadDelta( sideB ? Bodies::JointA( joint ) : Bodies::JointB( joint ), dpOther, dqOther );
	b2Vec2 P;
	float LA, LB;
	bool active = sideB ? JointWarmStartTerms( joint, dqOther, dpOther, dq, dp, P, LA, LB )
						: JointWarmStartTerms( joint, dq, dp, dqOther, dpOther, P, LA, LB );
	if ( active == false )
	{
		return;
	}
	if ( sideB == false )
	{
		float mA = joint->invMassA, iA = joint->invIA;
		vx = vx - mA * P.x;
		vy = vy - mA * P.y;
		w -= iA * LA;
	}
	else
	{
		float mB = joint->invMassB, iB = joint->invIB;
		vx = vx + mB * P.x;
		vy = vy + mB * P.y;
		w += iB * LB;
	}
}

template <int kChunk = 4, typename Bodies>
B2G_DEVI void WarmStartBody( const ConstraintSoA& c, const JointSim* joints, const int* jointList, int overflowContactStart,
							 const int* list, int begin, int end, const Bodies& B, b2Rot dq, b2Vec2 dp, float& vx, float& vy,
							 float& w )
{
	// Entries go in chunks of kChunk: all of a chunk's constraint fields are gathered first
	// (independent loads), then applied in order.
	for ( int base = begin; base < end; base += kChunk )
	{
		int count = end - base < kChunk ? end - base : kChunk;
		int ent[kChunk];
#pragma unroll
		for ( int q = 0; q < kChunk; ++q )
		{
			ent[q] = q < count ? list[base + q] : 2; // padding reads as a joint entry and is skipped
		}

		float nX[kChunk], nY[kChunk], m[kChunk], iv[kChunk], roll[kChunk];
		float ni[kChunk][2], ti[kChunk][2], rx[kChunk][2], ry[kChunk][2];
		int points[kChunk];
#pragma unroll
		for ( int q = 0; q < kChunk; ++q )
		{
			if ( ent[q] & 2 )
			{
				continue;
			}
			int k = ent[q] >> 3;
			bool sideB = ( ent[q] & 1 ) != 0;
			bool overflow = k >= overflowContactStart;
			nX[q] = c.f[kcNormalX][k];
			nY[q] = c.f[kcNormalY][k];
			m[q] = sideB ? c.f[kcInvMassB][k] : c.f[kcInvMassA][k];
			iv[q] = sideB ? c.f[kcInvIB][k] : c.f[kcInvIA][k];
			roll[q] = c.f[kcRollingImpulse][k];
			points[q] = overflow ? c.pointCount[k] : 2;
#pragma unroll
			for ( int j = 0; j < 2; ++j )
			{
				int o = j == 0 ? 0 : ( kcAnchorA2X - kcAnchorA1X );
				ni[q][j] = c.f[kcNormalImpulse1 + o][k];
				ti[q][j] = c.f[kcTangentImpulse1 + o][k];
				rx[q][j] = sideB ? c.f[kcAnchorB1X + o][k] : c.f[kcAnchorA1X + o][k];
				ry[q][j] = sideB ? c.f[kcAnchorB1Y + o][k] : c.f[kcAnchorA1Y + o][k];
			}
		}

#pragma unroll
		for ( int q = 0; q < kChunk; ++q )
		{
			if ( q >= count )
			{
				break;
			}
			int entry = ent[q];
			bool sideB = ( entry & 1 ) != 0;
			if ( entry & 2 )
			{
				WarmStartJointSide( joints + jointList[entry >> 3], sideB, B, dq, dp, vx, vy, w );
				continue;
			}
			bool overflow = ( entry >> 3 ) >= overflowContactStart;
			// the wide lanes form the tangent as 0 - nX, the scalar overflow solver as -nX
			float tX = nY[q];
			float tY = overflow ? -nX[q] : 0.0f - nX[q];
#pragma unroll
			for ( int j = 0; j < 2; ++j )
			{
				if ( j >= points[q] )
				{
					break;
				}
				float Px = ni[q][j] * nX[q] + ti[q][j] * tX;
				float Py = ni[q][j] * nY[q] + ti[q][j] * tY;
				if ( sideB == false )
				{
					w = w - iv[q] * ( rx[q][j] * Py - ry[q][j] * Px );
					vx = vx - m[q] * Px;
					vy = vy - m[q] * Py;
				}
				else
				{
					w = w + iv[q] * ( rx[q][j] * Py - ry[q][j] * Px );
					vx = vx + m[q] * Px;
					vy = vy + m[q] * Py;
				}
			}
			w = sideB ? w + iv[q] * roll[q] : w - iv[q] * roll[q];
		}
	}

	// total normal impulses, once per contact (kept out of the loop above so its loads carry no
	// dependence on stores)
	for ( int e = begin; e < end; ++e )
	{
		int entry = list[e];
		if ( ( entry & 6 ) != 4 )
		{
			continue;
		}
		int k = entry >> 3;
		int points = k >= overflowContactStart ? c.pointCount[k] : 2;
		for ( int j = 0; j < points; ++j )
		{
			int o = j == 0 ? 0 : ( kcAnchorA2X - kcAnchorA1X );
			c.f[kcTotalNormalImpulse1 + o][k] = c.f[kcTotalNormalImpulse1 + o][k] + c.f[kcNormalImpulse1 + o][k];
		}
	}
}

} // namespace b2g
