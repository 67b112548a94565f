// Double-tiling phase with one wave per 16 x 16-site block, for lattices with
// too few blocks to fill the chip with one lane per block.
//
// dt_phase_kernel gives a block to one lane, which does its 256 updates one
// after the other, an LDS round trip each: 22-25 us per phase however few
// blocks there are (256 blocks at 512^2 are four waves on 1024 SIMDs).  Here
// the 64 lanes of a wave draw the 256 updates of a block together (the stream
// jumped to every lane's draws), find out which of them may be done at the
// same time, and do these together on the block's bit rows.
//
// Two updates of a block touch common slopes only if their sites are the same
// or next neighbours.  A window of 64 consecutive updates (one per lane) is
// therefore cut into levels: an update's level is one more than the highest
// level among the earlier updates of the window on its own or a neighbouring
// site.  Updates of one level touch disjoint slopes, and every update comes
// after all earlier ones that it depends on, so applying level after level,
// window after window gives the sequential result bit for bit.  An update
// that accepts neither a minimum nor a maximum changes nothing and is left
// out.  Random sites need 4.3 levels per window, 17 (12 to 25) per block, against
// 256 sequential steps.
//
// What bounds it: latency (the lattice and stream loads, the LDS round trips
// of the level search, some 17 dependent steps of 9 instructions) on small
// lattices; from 4096^2 on VALU issue (about 700 instructions per block) and the
// LDS (random 8-byte accesses, 28 per block and lane).  Tried and not kept: four
// blocks per wave, levelled one after the other and applied together by 16
// lanes each (4096^2 106 us per MCS against 91 then: twice the registers and
// LDS).
#include "kpz_kernels.hpp"

namespace kpz {

namespace {

constexpr int DW_WAVES = 4;                  // blocks per workgroup
constexpr int DW_PITCH = 17;                 // sites of a row and one empty column between rows
constexpr int DW_SITES = 18 * DW_PITCH;      // 16 rows with an empty row below and above
constexpr int DW_LEVELS = 32;                // levels applied per pass
constexpr int DW_LPITCH = DW_LEVELS + 4;     // words per row of the level table (16-byte aligned rows)
static_assert(16 * DW_LPITCH * 4 <= 2 * DW_SITES * 8, "the level table reuses the window masks");

// bits 0,2,..,30 -> 0..15
__device__ __forceinline__ uint32_t even_bits(uint32_t v)
{
	v &= 0x55555555u;
	v = (v | (v >> 1)) & 0x33333333u;
	v = (v | (v >> 2)) & 0x0F0F0F0Fu;
	v = (v | (v >> 4)) & 0x00FF00FFu;
	return (v | (v >> 8)) & 0x0000FFFFu;
}
// 0..15 -> bits 0,2,..,30
__device__ __forceinline__ uint32_t to_even_bits(uint32_t v)
{
	v &= 0xFFFFu;
	v = (v | (v << 8)) & 0x00FF00FFu;
	v = (v | (v << 4)) & 0x0F0F0F0Fu;
	v = (v | (v << 2)) & 0x33333333u;
	return (v | (v << 1)) & 0x55555555u;
}

// LDS accesses of a wave are done in the order they are issued; this keeps the
// compiler from exchanging those before and after
__device__ __forceinline__ void lds_in_order()
{
	__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
	__builtin_amdgcn_wave_barrier();
	__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// value of the next / previous lane within 16 lanes; the last / first lane gets `edge`
__device__ __forceinline__ uint32_t from_next(uint32_t v, uint32_t edge)
{
	return (uint32_t)__builtin_amdgcn_update_dpp((int)edge, (int)v, 0x101, 0xF, 0xF, false); // row_shl:1
}
__device__ __forceinline__ uint32_t from_prev(uint32_t v)
{
	return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, true); // row_shr:1
}

// UPD: 0 = KPZ (pqOneUpdate), 1 = pqSyncRngUpdate, 2 = disorder2SyncRngUpdate,
// 3 = EW; RO: random origin (as dt_phase_kernel)
// block i of nb, with this wave's LDS `masks`
template<int UPD, bool RO>
__device__ __forceinline__ void dt_wave_block(const DtPhaseArgs& a, const DtWaveJumps& J, int64_t i, int64_t nb,
                                              uint64_t* masks)
{
	const int lane = threadIdx.x & 63;

	// ---- the block's stream (dt_phase_kernel: DtSlcg::begin)
	const bool ownStream = a.T >= nb;
	const int64_t t = ownStream ? i : i % a.T;
	uint64_t s0 = a.st_in[t];
	if(!ownStream)
		s0 = a.jumps[i / a.T](s0);

	// ---- geometry, Kmc::DoubleTilingDD<2>::setBlock (inc/doubleTilingDD.h:71-78)
	const int lhx = a.lx - 5;
	const int ox = (int)((2 * (i & ((1ll << lhx) - 1)) + (a.ds & 1)) << 4) + a.sx;
	const int oy = (int)((2 * (i >> lhx) + (a.ds >> 1)) << 4) + a.sy;
	const int XW = 1 << (a.lx - 2);
	const int mXW = XW - 1, mYW = (1 << (a.ly - 2)) - 1;
	const int shx = RO ? (ox & 3) : 0;
	const int c0 = ox >> 2;

	// ---- lane r holds site row r: rows 0..15 of the block, 16 = the halo row
	// (its y slopes); further lanes repeat rows 0..15 and store nothing.  A site
	// row is one byte of each of five words: 20 sites, 17 of them from shx on.
	const int yr = oy + ((lane <= 16) ? lane : (lane & 15));
	const size_t rowWord = (size_t)((yr >> 2) & mYW) * XW;
	const int byte = yr & 3;
	uint32_t b[5];
#pragma unroll
	for(int k = 0; k < 5; ++k)
		b[k] = a.lat[rowWord + ((c0 + k) & mXW)];
	{
		// no update yet on any site of any window
		uint4* z = reinterpret_cast<uint4*>(masks);
#pragma unroll
		for(int k = 0; k < (2 * DW_SITES * 8 / 16 + 63) / 64; ++k)
			if(64 * k + lane < 2 * DW_SITES * 8 / 16)
				z[64 * k + lane] = make_uint4(0, 0, 0, 0);
	}

	// ---- the updates: lane l draws updates l, 64 + l, 128 + l, 192 + l
	uint64_t s = s0;
#pragma unroll
	for(int k = 0; k < 6; ++k)
	{
		const uint64_t j = J.lane[k](s);
		s = ((lane >> k) & 1) ? j : s;
	}
	uint32_t mask[4]; // bit x: a minimum is accepted, bit 16 + x: a maximum
	int row[4], at[4];
	bool live[4];
#pragma unroll
	for(int w = 0; w < 4; ++w)
	{
		uint64_t u = a.step(s);
		const uint32_t r1 = slcg_fold(u);
		u = a.step(u);
		const uint32_t r2 = slcg_fold(u);
		const int x = RO ? (int)((r1 >> 19) & 15) : (int)(r1 >> 28);
		const int y = RO ? (int)((r2 >> 19) & 15) : (int)(r2 >> 28);
		bool mn = true, mx = UPD != 0;
		if constexpr(UPD == 1 || UPD == 2)
		{
			u = a.step(u);
			const uint32_t r23 = slcg_fold(u) & 0x7FFFFFu;
			uint32_t tp = a.tp, tq = a.tq;
			if constexpr(UPD == 2)
			{
				const int dx = ox + x, dy = oy + y;
				const uint32_t dw = a.dis[(size_t)((dy >> 2) & mYW) * XW + ((dx >> 2) & mXW)];
				const uint32_t cls = (dw >> (8 * (dy & 3) + 2 * (dx & 3))) & 3u;
				tp = (cls & 2) ? ((cls & 1) ? a.tpc[3] : a.tpc[2]) : ((cls & 1) ? a.tpc[1] : a.tpc[0]);
				tq = (cls & 2) ? ((cls & 1) ? a.tqc[3] : a.tqc[2]) : ((cls & 1) ? a.tqc[1] : a.tqc[0]);
			}
			mn = r23 < tp;
			mx = r23 < tq;
		}
		mask[w] = (mn ? 1u << x : 0u) | (mx ? 0x10000u << x : 0u);
		live[w] = mn || mx;
		row[w] = y;
		at[w] = (y + 1) * DW_PITCH + x + 1;
		s = J.window(s);
	}

	// ---- earlier updates of the window on the own or a neighbouring site, two
	// windows at a time (5 KB of LDS per wave, so that 8 waves fit a SIMD)
	uint64_t before[4];
	const uint64_t earlier = (1ull << lane) - 1;
	lds_in_order();
#pragma unroll
	for(int w0 = 0; w0 < 4; w0 += 2)
	{
#pragma unroll
		for(int k = 0; k < 2; ++k)
			if(live[w0 + k])
				__hip_atomic_fetch_or(&masks[k * DW_SITES + at[w0 + k]], 1ull << lane, __ATOMIC_RELAXED,
				                      __HIP_MEMORY_SCOPE_WAVEFRONT);
		lds_in_order();
#pragma unroll
		for(int k = 0; k < 2; ++k)
		{
			const uint64_t* m = masks + k * DW_SITES + at[w0 + k];
			before[w0 + k] = (m[0] | m[-1] | m[1] | m[-DW_PITCH] | m[DW_PITCH]) & earlier;
		}
		lds_in_order();
		if(w0 == 0)
		{
			masks[at[0]] = 0;
			masks[DW_SITES + at[1]] = 0;
			lds_in_order();
		}
	}

	// ---- levels: an update waits while one of those has not been done
	int level[4] = {0, 0, 0, 0}, depth[4] = {0, 0, 0, 0};
	uint64_t todo[4];
#pragma unroll
	for(int w = 0; w < 4; ++w)
		todo[w] = __ballot(live[w]);
	while((todo[0] | todo[1] | todo[2] | todo[3]) != 0)
	{
#pragma unroll
		for(int w = 0; w < 4; ++w)
		{
			// an update that is not in todo any more has nothing before it there
			const bool waits = (before[w] & todo[w]) != 0;
			depth[w] += todo[w] != 0;
			todo[w] &= __ballot(waits);
			level[w] += waits;
		}
	}
	int total = 0;
#pragma unroll
	for(int w = 0; w < 4; ++w)
	{
		level[w] += total;
		total += depth[w];
	}

	// ---- bit rows: X = columns 0..16 (16 = the halo column), Y = columns 0..15
	uint64_t raw = 0; // 20 sites, 2 bits each
#pragma unroll
	for(int k = 0; k < 5; ++k)
		raw |= (uint64_t)((b[k] >> (8 * byte)) & 0xFFu) << (8 * k);
	uint32_t X, Y;
	{
		const uint64_t v = raw >> (2 * shx);
		X = even_bits((uint32_t)v) | (((uint32_t)(v >> 32) & 1u) << 16);
		Y = even_bits((uint32_t)v >> 1);
	}
	// y slopes of the halo row: lane 15's upper neighbour
	uint32_t top = (uint32_t)__builtin_amdgcn_readlane((int)Y, 16);

	uint32_t* const table = reinterpret_cast<uint32_t*>(masks); // [row][level]
	for(int base = 0; base < total; base += DW_LEVELS)
	{
		{
			uint4* z = reinterpret_cast<uint4*>(table);
#pragma unroll
			for(int k = 0; k < (16 * DW_LPITCH / 4 + 63) / 64; ++k)
				if(64 * k + lane < 16 * DW_LPITCH / 4)
					z[64 * k + lane] = make_uint4(0, 0, 0, 0);
		}
		lds_in_order();
#pragma unroll
		for(int w = 0; w < 4; ++w)
		{
			const int l = level[w] - base;
			if(live[w] && l >= 0 && l < DW_LEVELS)
				__hip_atomic_fetch_or(&table[row[w] * DW_LPITCH + l], mask[w], __ATOMIC_RELAXED,
				                      __HIP_MEMORY_SCOPE_WAVEFRONT);
		}
		lds_in_order();
		const int n = min(DW_LEVELS, total - base);
		const uint4* mine = reinterpret_cast<const uint4*>(table + (lane & 15) * DW_LPITCH);
		uint4 next = mine[0];
		for(int l = 0; l < n; l += 4) // levels past the last one are empty
		{
			const uint32_t m[4] = {next.x, next.y, next.z, next.w};
			next = mine[min(l / 4 + 1, DW_LEVELS / 4)]; // the last row entry is padding
#pragma unroll
			for(int k = 0; k < 4; ++k)
			{
				// as the update of dt_block, for all sites of the level: a minimum
				// has own X = 0, right X = 1, own Y = 0, up Y = 1, a maximum the
				// opposite; its flip is X - m (X + m), Y and the Y above toggle
				const uint32_t up = from_next(Y, top);
				const uint32_t rx = X >> 1;
				if constexpr(UPD == 0)
				{
					const uint32_t f = rx & ~X & ~Y & up & m[k];
					X -= f;
					top ^= f; // lane 15's own
					Y ^= f;
					Y ^= from_prev(f);
				}
				else
				{
					const uint32_t fn = rx & ~X & ~Y & up & (m[k] & 0xFFFFu);
					const uint32_t fx = ~rx & X & Y & ~up & (m[k] >> 16);
					const uint32_t f = fn | fx;
					X = X - fn + fx;
					top ^= f;
					Y ^= f;
					Y ^= from_prev(f);
				}
			}
		}
		lds_in_order();
	}

	// ---- back to bytes.  No other lane of the launch writes the words the
	// block touches, so a row is stored byte by byte.
	const uint32_t newTop = (uint32_t)__builtin_amdgcn_readlane((int)top, 15);
	uint64_t own; // bits of the 20 sites that belong to the block's row
	if(lane < 16)
		own = 0x1FFFFFFFFull << (2 * shx);
	else
	{
		own = 0xAAAAAAAAull << (2 * shx);
		Y = newTop;
	}
	const uint64_t v = (((uint64_t)(X >> 16) & 1u) << 32 | to_even_bits(X) | to_even_bits(Y) << 1) << (2 * shx);
	const uint64_t out = (raw & ~own) | (v & own);
	if(lane <= 16)
	{
		uint8_t* p = reinterpret_cast<uint8_t*>(a.lat) + byte;
#pragma unroll
		for(int k = 0; k < 5; ++k)
			if((own >> (8 * k)) & 0xFFu)
				p[4 * (rowWord + ((c0 + k) & mXW))] = (uint8_t)(out >> (8 * k));
	}
	if(lane == 0 && (ownStream || i + a.T >= nb))
		a.st_out[t] = a.blockJ(s0);
}

template<int UPD, bool RO>
__global__ __launch_bounds__(64 * DW_WAVES) void dt_wave_kernel(DtPhaseArgs a, DtWaveJumps J, int64_t nb)
{
	__shared__ __align__(16) uint64_t masks[DW_WAVES][2 * DW_SITES];
	const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
	const int64_t i = (int64_t)blockIdx.x * DW_WAVES + wave;
	if(i >= nb)
		return; // whole wave; no barrier in this kernel
	dt_wave_block<UPD, RO>(a, J, i, nb, masks[wave]);
}

// One DT phase of every DT (DTr: RO) replica of a batch: entry of the lane
// table -> wave (batch_dt_kernel takes a lane for each)
template<bool RO>
__global__ __launch_bounds__(64 * DW_WAVES) void batch_dt_wave_kernel(BatchDtArgs a)
{
	__shared__ __align__(16) uint64_t masks[DW_WAVES][2 * DW_SITES];
	const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
	const int64_t e = (int64_t)blockIdx.x * DW_WAVES + wave + (RO ? a.nstatic : 0);
	if(e >= (RO ? a.nlanes : a.nstatic))
		return; // whole wave, here and below
	const uint2 w = a.lanes[e];
	if(w.x == 0xFFFFFFFFu || (a.limit && a.m >= a.limit[w.x]))
		return;
	const BatchRep& rep = a.reps[w.x];
	DtPhaseArgs p{};
	p.lat = rep.lat;
	p.lx = rep.lx;
	p.ly = rep.ly;
	p.st_in = p.st_out = rep.st[0];
	p.step = rep.step;
	p.blockJ = rep.full;
	p.tp = rep.tp;
	p.tq = rep.tq;
	const size_t mi = (size_t)a.m * a.nreps + w.x;
	p.ds = (a.order[mi] >> (2 * a.d)) & 3;
	if constexpr(RO)
	{
		const uint16_t sh = a.shift[mi];
		p.sx = sh & 0xFF;
		p.sy = sh >> 8;
	}
	const int64_t nb = 1ll << (rep.lx + rep.ly - 10);
	p.T = nb;
	// dt_wave_jumps on the scalar unit
	DtWaveJumps J;
	J.lane[0] = compose(rep.step, rep.step);
	if(rep.mode)
		J.lane[0] = compose(rep.step, J.lane[0]);
#pragma unroll
	for(int k = 1; k < 6; ++k)
		J.lane[k] = compose(J.lane[k - 1], J.lane[k - 1]);
	J.window = compose(J.lane[5], J.lane[5]);
	if(rep.mode)
		dt_wave_block<1, RO>(p, J, w.y, nb, masks[wave]);
	else
		dt_wave_block<0, RO>(p, J, w.y, nb, masks[wave]);
}

template<int UPD>
void launch(const DtPhaseArgs& a, const DtWaveJumps& J, int64_t nb, hipStream_t stream)
{
	const dim3 grid((unsigned)((nb + DW_WAVES - 1) / DW_WAVES));
	if(a.random_origin)
		hipLaunchKernelGGL((dt_wave_kernel<UPD, true>), grid, dim3(64 * DW_WAVES), 0, stream, a, J, nb);
	else
		hipLaunchKernelGGL((dt_wave_kernel<UPD, false>), grid, dim3(64 * DW_WAVES), 0, stream, a, J, nb);
}

} // namespace

bool dt_wave_better(int lbx, int lby, int64_t nb, int upd, bool tinyMT)
{
	return lbx == 4 && lby == 4 && !tinyMT && nb <= (upd == 2 ? 1 << 14 : 1 << 13);
}

DtWaveJumps dt_wave_jumps(const Affine& step, int drawsPerUpdate)
{
	DtWaveJumps J;
	Affine j = affine_pow(step, (uint64_t)drawsPerUpdate);
	for(int k = 0; k < 6; ++k)
	{
		J.lane[k] = j;
		j = compose(j, j);
	}
	J.window = j;
	return J;
}

hipError_t launch_dt_wave(const DtPhaseArgs& a, const DtWaveJumps& J, hipStream_t stream)
{
	if(a.lbx != 4 || a.lby != 4 || a.tmt || a.T < 1 || (a.upd == 2 && !a.dis))
		return hipErrorInvalidValue;
	const int64_t nb = 1ll << (a.lx + a.ly - 10);
	if(a.T < nb && !a.jumps)
		return hipErrorInvalidValue;
	switch(a.upd)
	{
		case 0: launch<0>(a, J, nb, stream); break;
		case 1: launch<1>(a, J, nb, stream); break;
		case 2: launch<2>(a, J, nb, stream); break;
		case 3: launch<3>(a, J, nb, stream); break;
		default: return hipErrorInvalidValue;
	}
	return hipGetLastError();
}

hipError_t launch_batch_dt_wave(const BatchDtArgs& a, hipStream_t stream)
{
	if(a.nstatic < 0 || a.nstatic > a.nlanes)
		return hipErrorInvalidValue;
	auto grid = [](int64_t n) { return dim3((unsigned)((n + DW_WAVES - 1) / DW_WAVES)); };
	if(a.nstatic > 0)
		hipLaunchKernelGGL(batch_dt_wave_kernel<false>, grid(a.nstatic), dim3(64 * DW_WAVES), 0, stream, a);
	if(a.nlanes > a.nstatic)
		hipLaunchKernelGGL(batch_dt_wave_kernel<true>, grid(a.nlanes - a.nstatic), dim3(64 * DW_WAVES), 0, stream, a);
	return hipGetLastError();
}

} // namespace kpz
