// One whole SCABit MCS (both half-sweeps, modes 0 and 1 of cbbit_half_kernel)
// in one pass over the lattice.
//
// The bit-parallel half-sweep is bound by memory: each of the two reads and
// writes every word (1 byte per site update in all) for a few instructions per
// site.  Here the lanes of a row walk upwards and do the second half-sweep of a
// row as soon as the first one has passed the rows around it, so every word is
// read once and written once per MCS: 65536^2 takes 441 us (788 in two
// half-sweeps), 4.9 TB/s, what a copy of that size reaches; 16384^2 25 us (45),
// 8192^2 9.6 (15), and on small lattices one launch instead of two, 2048^2 4.9
// (6.6).  The per-site rule gains where its own half-sweeps come close to the
// memory rate (cbbit_mcs_better).
//
// Half-sweep s acts on the sites of sublattice s.  On row y it flips bits of
// X_s(y), Y_s(y), X_o(y) and Y_o(y + 1) (o the other sublattice), each bit
// belonging to one active site only.  The second half-sweep of row y - 1
// therefore needs the first one of rows y - 2, y - 1 and y, and a band of rows
// [y0, y1) needs the first half-sweep of rows y0 - 2 .. y1 and the second one
// of rows y0 - 1 .. y1 - 1; rows outside the band are computed again (2 / R of
// the work for R rows) and not stored.  Along x a site's right neighbour lies
// in the next bit on every other row; a band spans the whole row, so that the
// bits that cross from word to word stay inside it.  Source and destination are
// different lattices, since neighbouring bands read each other's rows.
#include "kpz_kernels.hpp"

#include "kpz_draws.hpp"

namespace kpz {

namespace {

__device__ __forceinline__ uint32_t lane_value(uint32_t v, int src, int width)
{
	return (uint32_t)__shfl((int)v, src, width);
}

// the two draws of a word from the state before them, pSyncRngUpdateVL3
// (kpz/schedulerCPUCBBit_nested.inl:240)
__device__ __forceinline__ uint64_t vl3_word(uint64_t& u, const Affine& step)
{
	u = step(u);
	const uint64_t hi = slcg_fold(u);
	u = step(u);
	return (hi << 32) ^ (uint64_t)slcg_fold(u);
}

// the worker of a row and the row's index among the worker's rows
struct RowWorker {
	int t, r;
	__device__ __forceinline__ RowWorker(int y, int per, int rem)
	{
		const int big = rem * (per + 1);
		if(y < big)
		{
			t = y / (per + 1);
			r = y - t * (per + 1);
		}
		else
		{
			t = rem + (y - big) / per;
			r = (y - big) - (t - rem) * per;
		}
	}
	__device__ __forceinline__ void next(int per, int rem, int T)
	{
		if(++r == per + (t < rem ? 1 : 0))
		{
			r = 0;
			t = (t + 1 == T) ? 0 : t + 1;
		}
	}
};

// Rows of up to 64 words: a group of Wn lanes per band, a word per lane.
__global__ __launch_bounds__(256) void cbbit_mcs_narrow_kernel(CbMcsArgs a)
{
	const int lane = threadIdx.x & 63;
	const int Y = 1 << a.ly, lW = a.lx - 7, Wn = 1 << lW, R = 1 << a.lR;
	const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
	int band = (int)(gid >> lW);
	const bool keep = band < (Y >> a.lR);
	band = keep ? band : 0; // spare lanes of the last wave follow band 0
	const int w = lane & (Wn - 1);
	const int gUp = (lane + 1) & (Wn - 1), gDn = (lane - 1) & (Wn - 1);
	const uint64_t* __restrict__ src = (const uint64_t*)a.src;
	uint64_t* __restrict__ dst = (uint64_t*)a.dst;
	const size_t Q = (size_t)Wn << a.ly;
	const Affine J = a.wordJ[w], step = a.step;

	const int y0 = band << a.lR;
	int y = (y0 - 2) & (Y - 1);
	RowWorker wk(y, a.per, a.rem);
	const bool single = a.per == 1 && a.rem == 0; // a worker per row
	auto row = [&](int yy) { return (size_t)(yy & (Y - 1)) * Wn + w; };
	auto random = [&](uint64_t start) {
		uint64_t u = J(start);
		return vl3_word(u, step);
	};
	auto right = [&](uint64_t v) { return (v >> 1) | ((uint64_t)lane_value((uint32_t)v, gUp, Wn) << 63); };
	auto left = [&](uint64_t f) { return (f << 1) | (lane_value((uint32_t)(f >> 32), gDn, Wn) >> 31); };

	uint64_t x0 = src[row(y)], v0 = src[Q + row(y)], x1 = src[2 * Q + row(y)], v1up = src[3 * Q + row(y + 1)];
	uint64_t px0 = 0, pv0 = 0, px1 = 0, pv1 = 0, v1 = 0; // row y - 1 and Y_1(y)
	uint64_t st = a.st_in[wk.t], start1 = 0;             // start1: second half-sweep's stream start of row y - 1
	for(int i = 0; i < R + 3; ++i)
	{
		// the next row's words and stream, in flight during this row's work
		uint64_t nx0 = 0, nv0 = 0, nx1 = 0, nv1 = 0;
		RowWorker nk = wk;
		nk.next(a.per, a.rem, a.T);
		const uint64_t nst = a.st_in[nk.t];
		if(i < R + 2)
		{
			const size_t o = row(y + 1);
			nx0 = src[o];
			nv0 = src[Q + o];
			nx1 = src[2 * Q + o];
			nv1 = src[3 * Q + row(y + 2)];
		}

		const Affine full = (wk.t < a.rem) ? a.fullBig : a.fullSmall;
		uint64_t s0 = st, s1 = full(st);
		if(keep && wk.r == 0 && w == 0 && i >= 2 && i < R + 2)
			a.st_out[wk.t] = full(s1);
		if(!single)
		{
			const Affine rj = a.rowJ[wk.r];
			s0 = rj(s0);
			s1 = rj(s1);
		}
		// y0 is even: on even rows the first half-sweep, and on the odd rows below
		// them the second one, find the right neighbour in the same bit
		const bool par = !(i & 1);
		// first half-sweep, row y
		{
			const uint64_t xs = par ? x1 : right(x1);
			const uint64_t f = ~(x0 | v0) & xs & v1up & random(s0);
			x0 ^= f;
			v0 ^= f;
			v1up ^= f;
			x1 ^= par ? f : left(f);
		}
		// second half-sweep, row y - 1
		if(i >= 2)
		{
			const uint64_t xs = par ? px0 : right(px0);
			const uint64_t f = ~(px1 | pv1) & xs & v0 & random(start1);
			px1 ^= f;
			pv1 ^= f;
			v0 ^= f;
			px0 ^= par ? f : left(f);
			if(keep && i >= 3)
			{
				const size_t o = row(y - 1);
				dst[o] = px0;
				dst[Q + o] = pv0;
				dst[2 * Q + o] = px1;
				dst[3 * Q + o] = pv1;
			}
		}
		px0 = x0;
		pv0 = v0;
		px1 = x1;
		pv1 = v1;
		v1 = v1up;
		start1 = s1;
		x0 = nx0;
		v0 = nv0;
		x1 = nx1;
		v1up = nv1;
		st = nst;
		wk = nk;
		y = (y + 1) & (Y - 1);
	}
}

// Rows of 128 words and more: a band per workgroup of Wn / 2 lanes (MULTI), or
// per wave for 128 words; a lane holds two neighbouring words, whose draws
// follow each other in the stream (one jump for both).  The bits that cross
// from wave to wave, all of them on odd steps, go through LDS, with two
// barriers per two rows.
struct Words {
	uint64_t a, b;
};
__device__ __forceinline__ Words load2(const uint64_t* p)
{
	const ulonglong2 v = *reinterpret_cast<const ulonglong2*>(p);
	return {v.x, v.y};
}
__device__ __forceinline__ void store2(uint64_t* p, const Words& v)
{
	*reinterpret_cast<ulonglong2*>(p) = make_ulonglong2(v.a, v.b);
}

// NT: 0 = bit-parallel, else per site with 1 (q = 0) or 2 thresholds per draw
template<int NT, bool MULTI>
__global__ __launch_bounds__(MULTI ? 1024 : 256) void cbbit_mcs_wide_kernel(CbMcsArgs a)
{
	__shared__ uint32_t low[16], high[16]; // per wave: bits for the wave before / after
	const int lane = threadIdx.x & 63;
	const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
	const int nw = MULTI ? (int)blockDim.x >> 6 : 1;
	const int Y = 1 << a.ly, Wn = 1 << (a.lx - 7), R = 1 << a.lR;
	const int band = MULTI ? (int)blockIdx.x : (int)blockIdx.x * 4 + wv;
	if(!MULTI && band >= (Y >> a.lR))
		return; // whole wave; no barrier in this variant
	const int w = 2 * (MULTI ? (int)threadIdx.x : lane);
	const uint64_t* __restrict__ src = (const uint64_t*)a.src;
	uint64_t* __restrict__ dst = (uint64_t*)a.dst;
	const size_t Q = (size_t)Wn << a.ly;
	const Affine J = a.wordJ[w], step = a.step;

	const int y0 = band << a.lR;
	int y = (y0 - 2) & (Y - 1);
	RowWorker wk(y, a.per, a.rem);
	const bool single = a.per == 1 && a.rem == 0;
	auto row = [&](int yy) { return (size_t)(yy & (Y - 1)) * Wn + w; };
	// sites that flip if they are a minimum (p) or a maximum (q), from the
	// row's stream start
	struct Accept {
		Words p, q;
	};
	auto accept = [&](uint64_t start) {
		uint64_t u = J(start);
		Accept r{{0, 0}, {0, 0}};
		if constexpr(NT == 0)
		{
			r.p.a = vl3_word(u, step);
			r.p.b = vl3_word(u, step);
		}
		else
		{
			uint32_t lo = (uint32_t)u, h24 = (uint32_t)(u >> 32);
#pragma unroll 1
			for(int k = 0; k < 2; ++k) // the second word's draws follow the first one's
			{
				uint64_t pb = 0, qb = 0, none = 0;
				cbbit_word_draws<uint64_t, NT>(lo, h24, step, a.tp, a.tq, 0, 0, pb, qb, none, none);
				r.p = {r.p.b, pb};
				r.q = {r.q.b, qb};
			}
		}
		return r;
	};
	// first bit of the next lane / last bit of the lane before, within the wave
	auto next_bit = [&](uint64_t firstWord) { return lane_value((uint32_t)firstWord, (lane + 1) & 63, 64) & 1u; };
	auto prev_bit = [&](uint64_t lastWord) { return lane_value((uint32_t)(lastWord >> 32), (lane - 1) & 63, 64) >> 31; };
	auto right = [&](const Words& v, uint32_t in) {
		return Words{(v.a >> 1) | (v.b << 63), (v.b >> 1) | ((uint64_t)in << 63)};
	};
	auto left = [&](const Words& f, uint32_t in) { return Words{(f.a << 1) | in, (f.b << 1) | (f.a >> 63)}; };
	auto flips = [&](const Words& x, const Words& v, const Words& xs, const Words& up, const Accept& r) {
		Words f{~(x.a | v.a) & xs.a & up.a & r.p.a, ~(x.b | v.b) & xs.b & up.b & r.p.b};
		if constexpr(NT == 2)
		{
			f.a |= x.a & v.a & ~(xs.a | up.a) & r.q.a;
			f.b |= x.b & v.b & ~(xs.b | up.b) & r.q.b;
		}
		return f;
	};
	auto flip = [&](Words& v, const Words& f) {
		v.a ^= f.a;
		v.b ^= f.b;
	};
	auto barrier = [&]() {
		if constexpr(MULTI) // the loads in flight need not be waited for
			asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
	};

	Words x0 = load2(src + row(y)), v0 = load2(src + Q + row(y)), x1 = load2(src + 2 * Q + row(y)),
	      v1up = load2(src + 3 * Q + row(y + 1));
	Words px0{0, 0}, pv0{0, 0}, px1{0, 0}, pv1{0, 0}, v1{0, 0}; // row y - 1 and Y_1(y)
	Words nx0, nv0, nx1, nv1;                                   // the next row
	uint64_t st = a.st_in[wk.t], nst = 0, start1 = 0, s0 = 0, s1 = 0;
	RowWorker nk = wk;
	auto fetch = [&](int i) {
		nk.next(a.per, a.rem, a.T);
		nst = a.st_in[nk.t];
		if(i < R + 2)
		{
			nx0 = load2(src + row(y + 1));
			nv0 = load2(src + Q + row(y + 1));
			nx1 = load2(src + 2 * Q + row(y + 1));
			nv1 = load2(src + 3 * Q + row(y + 2));
		}
		const Affine full = (wk.t < a.rem) ? a.fullBig : a.fullSmall;
		s0 = st;
		s1 = full(st);
		if(wk.r == 0 && w == 0 && i >= 2 && i < R + 2)
			a.st_out[wk.t] = full(s1);
		if(!single)
		{
			const Affine rj = a.rowJ[wk.r];
			s0 = rj(s0);
			s1 = rj(s1);
		}
	};
	auto store = [&]() {
		const size_t o = row(y - 1);
		store2(dst + o, px0);
		store2(dst + Q + o, pv0);
		store2(dst + 2 * Q + o, px1);
		store2(dst + 3 * Q + o, pv1);
	};
	auto advance = [&]() {
		px0 = x0;
		pv0 = v0;
		px1 = x1;
		pv1 = v1;
		v1 = v1up;
		start1 = s1;
		x0 = nx0;
		v0 = nv0;
		x1 = nx1;
		v1up = nv1;
		st = nst;
		wk = nk;
		y = (y + 1) & (Y - 1);
	};
	for(int i = 0;; i += 2)
	{
		// even step (y0 is even): the right neighbours of the first half-sweep on
		// row y and of the second one on row y - 1 are in the same bit
		fetch(i);
		{
			const Words f = flips(x0, v0, x1, v1up, accept(s0));
			flip(x0, f);
			flip(v0, f);
			flip(v1up, f);
			flip(x1, f);
		}
		if(i >= 2)
		{
			const Words f = flips(px1, pv1, px0, v0, accept(start1));
			flip(px1, f);
			flip(pv1, f);
			flip(v0, f);
			flip(px0, f);
			if(i >= 4)
				store();
		}
		if(i == R + 2)
			return;
		advance();
		// odd step: they are in the next bit.  px0 is row y - 1's X_0 after the
		// first half-sweep, x1 row y's X_1 before it
		uint32_t inX1 = next_bit(x1.a), inX0 = next_bit(px0.a);
		if constexpr(MULTI)
		{
			if(lane == 0)
				low[wv] = ((uint32_t)x1.a & 1u) | (((uint32_t)px0.a & 1u) << 1);
			barrier();
			if(lane == 63)
			{
				const uint32_t m = low[wv + 1 == nw ? 0 : wv + 1];
				inX1 = m & 1u;
				inX0 = m >> 1;
			}
		}
		fetch(i + 1);
		const Words f0 = flips(x0, v0, right(x1, inX1), v1up, accept(s0));
		flip(x0, f0);
		flip(v0, f0);
		flip(v1up, f0);
		Words f1{0, 0};
		if(i >= 2)
			f1 = flips(px1, pv1, right(px0, inX0), v0, accept(start1));
		uint32_t inF0 = prev_bit(f0.b), inF1 = prev_bit(f1.b);
		if constexpr(MULTI)
		{
			if(lane == 63)
				high[wv] = (uint32_t)(f0.b >> 63) | ((uint32_t)(f1.b >> 63) << 1);
			barrier();
			if(lane == 0)
			{
				const uint32_t m = high[wv == 0 ? nw - 1 : wv - 1];
				inF0 = m & 1u;
				inF1 = m >> 1;
			}
		}
		flip(x1, left(f0, inF0));
		if(i >= 2)
		{
			flip(px1, f1);
			flip(pv1, f1);
			flip(v0, f1);
			flip(px0, left(f1, inF1));
			store();
		}
		advance();
	}
}

} // namespace

// Bands of 64 rows, halved down to 2 rows while the launch has less than 2048
// waves.  us per MCS with targets of 1024 / 2048 / 8192 waves (8192: at least 4
// rows): 512^2 4.6 / 4.6 / 5.9, 4096^2 5.5 / 5.5 / 6.6, 8192^2 11.4 / 9.6 / 9.6,
// 16384^2 24.1 / 24.8 / 27.6, 32768^2 127 / 115 / 125, 65536^2 443 / 441 / 446.
// Narrow rows have several bands in a wave, whose rows lie a band apart: with
// 2^(lx - 7) words to a row a load takes only that part of each 128-byte line,
// and the caches of the XCDs lose the rest before the next rows want it.  Rows of
// up to 4 words take bands of 2 rows (256 x 2^18, 2 / 4 / 64 rows: 13.4 / 19.9 /
// 66.3 us per MCS; 512 x 2^17 11.3 / 13.4 / 51.7), rows of 8 words up to 32
// (1024 x 2^20, 32 / 64 rows: 172 / 214; x 2^22 679 / 665).
int cbbit_mcs_band(int lx, int ly, int mode)
{
	if(mode == 1)
		return ly < 5 ? ly : 5; // 65536^2: 962 us per MCS with 16 rows, 912 with 32, 923 with 64
	const int most = lx < 10 ? 1 : (lx == 10 ? 5 : 6);
	int lR = ly < most ? ly : most;
	const int lanes = lx <= 13 ? lx - 7 : lx - 8; // log2 lanes per band
	while(lR > 1 && ((1ll << (ly - lR + lanes)) >> 6) < 2048)
		--lR;
	return lR;
}

hipError_t launch_cbbit_mcs(const CbMcsArgs& a, hipStream_t stream)
{
	if(!a.src || !a.dst || a.src == a.dst || !a.wordJ || !a.rowJ || a.lx < 7 || a.lx > CBBIT_MCS_MAX_LX || a.ly < 1 ||
	   a.ly > 30 || a.lR < 1 || a.lR > a.ly || a.T < 1 || a.per < 1 || a.mode < 0 || a.mode > 1 ||
	   (a.mode == 1 && a.lx < 15))
		return hipErrorInvalidValue;
	const int64_t bands = 1ll << (a.ly - a.lR);
	const int lW = a.lx - 7;
	const dim3 wide((unsigned)(lW == 7 ? (bands + 3) / 4 : bands)), lanes(lW == 7 ? 256u : 1u << (lW - 1));
	if(a.mode == 1)
	{
		if(a.tq)
			hipLaunchKernelGGL((cbbit_mcs_wide_kernel<2, true>), wide, lanes, 0, stream, a);
		else
			hipLaunchKernelGGL((cbbit_mcs_wide_kernel<1, true>), wide, lanes, 0, stream, a);
	}
	else if(lW <= 6)
		hipLaunchKernelGGL(cbbit_mcs_narrow_kernel, dim3((unsigned)(((bands << lW) + 255) / 256)), dim3(256), 0, stream, a);
	else if(lW == 7)
		hipLaunchKernelGGL((cbbit_mcs_wide_kernel<0, false>), wide, lanes, 0, stream, a);
	else
		hipLaunchKernelGGL((cbbit_mcs_wide_kernel<0, true>), wide, lanes, 0, stream, a);
	return hipGetLastError();
}

} // namespace kpz
