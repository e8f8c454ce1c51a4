// Roots of unity exp(-2 pi i j / D) in FP32 for every denominator the transforms use, as
// constant device data: D = 2^a up to 8192 (the 4096-point stages and the 8192-cell real
// split) and D = 3 2^a up to 3072.  The D roots of one denominator are contiguous, at
// offset D (2^a) or D - 3 (3 2^a, in the second table): a stage's lanes read consecutive
// entries.  Values are computed at compile time in FP64 and rounded once.
//
// Bound: latency of one round of cached loads per kernel.  FP64 sincospi per twiddle in every
// kernel's prologue instead (14 to 22 calls per thread) measured: field of a 64x64 film 24.6 us
// against 20.3 with the tables, of a 1024x1024 film 109.3 against 92.6 us, RKDP54 step of
// 512x512x32 cells 4.34 against 4.26 ms; the results are the same bit for bit.
#pragma once

#include <hip/hip_runtime.h>

namespace bm {

constexpr int kTw2Max = 8192, kTw3Max = 3072;

// 16-byte aligned: entries are read 8 bytes at a time
struct alignas(16) Tw2Table { float v[2 * kTw2Max][2]; };
struct alignas(16) Tw3Table { float v[2 * kTw3Max - 3][2]; };

// cos and -sin of 2 pi j / D: the quarter turn nearest to j / D exactly, the rest (at most
// pi / 4) by the Taylor series (the terms left out are below 1e-18)
constexpr void tw_root(int j, int D, float out[2])
{
	const int q = (4 * j + D / 2) / D;                 // nearest quarter turn
	const double x = 6.283185307179586476925286766559 * (double)(4 * j - q * D) / (4.0 * (double)D), x2 = x * x;
	double c = 0, s = 0, tc = 1, ts = x;
	for (int n = 1; n < 20; n += 2) {
		c += tc; s += ts;
		tc *= -x2 / (double)(n * (n + 1));
		ts *= -x2 / (double)((n + 1) * (n + 2));
	}
	double re = c, im = s;
	switch (q & 3) {
	case 1: re = -s; im = c; break;
	case 2: re = -c; im = -s; break;
	case 3: re = s; im = -c; break;
	}
	out[0] = (float)re; out[1] = (float)-im;
}

constexpr Tw2Table make_tw2()
{
	Tw2Table t{};
	for (int D = 1; D <= kTw2Max; D *= 2) for (int j = 0; j < D; j++) tw_root(j, D, t.v[D + j]);
	return t;
}

constexpr Tw3Table make_tw3()
{
	Tw3Table t{};
	for (int D = 3; D <= kTw3Max; D *= 2) for (int j = 0; j < D; j++) tw_root(j, D, t.v[D - 3 + j]);
	return t;
}

static __device__ constexpr Tw2Table kTw2 = make_tw2();
static __device__ constexpr Tw3Table kTw3 = make_tw3();

// the roots of denominator D (2^a or 3 2^a): entry j is exp(-2 pi i j / D), 0 <= j < D
template <int D> __device__ __forceinline__ const float2* tw_roots()
{
	static_assert(alignof(Tw2Table) >= alignof(float2) && alignof(Tw3Table) >= alignof(float2), "entries are read as float2");
	static_assert(D >= 1 && ((D & (D - 1)) == 0 ? D <= kTw2Max : D % 3 == 0 && ((D / 3) & (D / 3 - 1)) == 0 && D <= kTw3Max), "no roots of this order");
	if constexpr ((D & (D - 1)) == 0) return reinterpret_cast<const float2*>(kTw2.v[D]);
	else return reinterpret_cast<const float2*>(kTw3.v[D - 3]);
}

} // namespace bm
