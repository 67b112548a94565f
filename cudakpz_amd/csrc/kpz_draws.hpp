// Device code shared by the kernels that draw from SLCG64 streams per site.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "kpz_common.hpp"

namespace kpz {

namespace {

// The high state word of an SLCG64 step mod 2^24: h aLo + lo aHi + carry, as
// two v_mad_u32_u24 (a[23:0] * b[23:0] + c) in one asm block.  Left to itself
// the compiler widens products used mod 2^23 to v_mul_lo_u32 + v_add3_u32;
// one block instead of two halves the wait states it pads asm blocks with.
__device__ __forceinline__ uint32_t hi24_step(uint32_t h, uint32_t aLo, uint32_t lo, uint32_t aHi, uint32_t carry)
{
	uint32_t r;
	asm("v_mad_u32_u24 %0, %3, %4, %5\n\tv_mad_u32_u24 %0, %1, %2, %0"
	    : "=&v"(r) : "v"(h), "v"(aLo), "v"(lo), "v"(aHi), "v"(carry));
	return r;
}

// Acceptance bits of 32 consecutive draws, draw k -> bit k.  The difference
// d = r - t of a draw's r < 2^23 (or 2^24) and a threshold t <= 2^23 (2^24)
// has bits 24..31 all equal to its sign, which is the acceptance r < t.  One
// v_bitop3 (a | (d & m)) copies that sign into any single bit m of those:
// draws 0-7, 8-15 and 16-23 go to bits 24-31 of three accumulators, shifted
// down once at the end, draws 24-31 straight to their own bits of a fourth.
// Three fast-class instructions per draw and threshold fewer slow ones than
// funnel-shifting the sign in (v_alignbit) and reversing the word.
struct SignBits32 {
	uint32_t a = 0, b = 0, c = 0, d = 0;
	template<int K>
	__device__ __forceinline__ void put(uint32_t diff)
	{
		static_assert(K >= 0 && K < 32, "draw index");
		constexpr uint32_t m = 1u << (24 + (K & 7));
		if constexpr(K < 8)
			a = __builtin_amdgcn_bitop3_b32(a, diff, m, 0xF8);
		else if constexpr(K < 16)
			b = __builtin_amdgcn_bitop3_b32(b, diff, m, 0xF8);
		else if constexpr(K < 24)
			c = __builtin_amdgcn_bitop3_b32(c, diff, m, 0xF8);
		else
			d = __builtin_amdgcn_bitop3_b32(d, diff, m, 0xF8);
	}
	__device__ __forceinline__ uint32_t bits() const { return (a >> 24) | (b >> 16) | (c >> 8) | d; }
};

// compile-time loop: f(integral_constant<int, K>) for K = 0..N-1
template<int N, int K = 0, class F>
__device__ __forceinline__ void static_for(F&& f)
{
	if constexpr(K < N)
	{
		f(std::integral_constant<int, K>{});
		static_for<N, K + 1>(f);
	}
}

// Wave priority around a run of random draws.  On gfx950 a SIMD issues two
// fast-class VALU instructions (plain logic, adds, right shifts) of different
// waves in one quad-cycle, but a slow-class one (multiplies, left shifts,
// compares) issues alone.  Left alone the waves of a SIMD spread over their
// draws (all slow) and their bit work (all fast) and few quad-cycles pair.
// With the draws of several sites in one run at high priority a wave leaves
// its slow part quickly and the waves gather in the fast part, where they
// pair: 64 v_mul_lo_u32 and 96 v_xor_b32 per round, 8 waves per SIMD, issue
// at 42.5 T lane-ops/s without and 52.4 T with the priorities.
__device__ __forceinline__ void draws_begin()
{
	__builtin_amdgcn_sched_barrier(0);
	__builtin_amdgcn_s_setprio(3);
	__builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ void draws_end()
{
	__builtin_amdgcn_sched_barrier(0);
	__builtin_amdgcn_s_setprio(0);
	__builtin_amdgcn_sched_barrier(0);
}

// Per-site acceptance bits of one SCABit word: the WB draws of the word from
// stream state (lo, h24), site k -> bit k of pb (minimum accepted: r23 < tp) and qb
// (maximum accepted: r23 < tq); NT = thresholds per draw: 1 (q = 0), 2 (p and
// q), 4 (two disorder classes: pb1, qb1 from tp1, tq1).  Only the low 23 bits
// of lo ^ hi are used: the low state word evolves on its own (lo' = A_lo lo +
// C mod 2^32) and hi' mod 2^24 needs only hi mod 2^24 and lo, so inside the
// word the high half is carried mod 2^24 with two 24-bit multiply-adds (the
// caller rebuilds the full state from the word's start by a jump).  The sign
// of r23 - t of every draw is copied into its own bit (SignBits32).
template<typename W, int NT>
__device__ __forceinline__ void cbbit_word_draws(uint32_t& lo, uint32_t& h24, const Affine& step, uint32_t tp, uint32_t tq,
                                                 uint32_t tp1, uint32_t tq1, W& pb, W& qb, W& pb1, W& qb1)
{
	const uint32_t aLo = (uint32_t)step.a, aHi = (uint32_t)(step.a >> 32);
	const uint64_t cc = step.c;
	static_for<(int)sizeof(W) / 4>([&](auto hc) {
		constexpr int h = decltype(hc)::value;
		SignBits32 P, Q, P1, Q1;
		// draws per run (draws_begin): 65536^2, p = .95, q = .05 takes 1.09 ms per
		// MCS without the runs, 1.00 with 4 or 8; at 32768^2 0.250 with 4, 0.253 with 8
		constexpr int U = 4;
		static_for<32 / U>([&](auto uc) {
			constexpr int k0 = decltype(uc)::value * U;
			uint32_t r[U];
			draws_begin();
#pragma unroll
			for(int i = 0; i < U; ++i)
			{
				const uint64_t pr = (uint64_t)lo * aLo + cc;
				h24 = hi24_step(h24, aLo, lo, aHi, (uint32_t)(pr >> 32));
				lo = (uint32_t)pr;
				r[i] = lo ^ h24;
			}
			draws_end();
			static_for<U>([&](auto kc) {
				constexpr int k = k0 + decltype(kc)::value;
				const uint32_t r23 = r[k - k0] & 0x7FFFFFu;
				P.template put<k>(r23 - tp);
				if constexpr(NT >= 2)
					Q.template put<k>(r23 - tq);
				if constexpr(NT == 4)
				{
					P1.template put<k>(r23 - tp1);
					Q1.template put<k>(r23 - tq1);
				}
			});
		});
		pb |= (W)P.bits() << (32 * h);
		qb |= (W)Q.bits() << (32 * h);
		if constexpr(NT == 4)
		{
			pb1 |= (W)P1.bits() << (32 * h);
			qb1 |= (W)Q1.bits() << (32 * h);
		}
	});
}

} // namespace

} // namespace kpz
