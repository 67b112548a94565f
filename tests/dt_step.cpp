// A double-tiling scheduler whose streams take any step s -> a s + c, also one
// that no skip of the generator gives (tests/test_gpu_dt_levels.py).
#include "kpz_scheduler.hpp"

#include <cstdio>

namespace {
struct Stepped : kpz::SchedulerDT {
	Stepped(int lx, int ly, bool ro, kpz::Affine step) : SchedulerDT(lx, ly, kpz::Params{}, ro) { step_ = step; }
};
} // namespace

// rule: 0 = mcs, 1 = mcsPQSyncRng, 2 = mcsDisorder2SyncRng (dis, class 1 with p1, q1), 3 = mcsEW
extern "C" int dt_step_run(int ro, int lx, int ly, uint64_t seed, uint64_t a, uint64_t c, int rule, double p, double q, double p1,
                           double q1, const uint32_t* dis, int n, uint32_t* lat, uint64_t* states)
{
	try
	{
		Stepped s(lx, ly, ro != 0, kpz::Affine{a, c});
		s.supplySeed(seed);
		s.initHomogeneous();
		s.setPQ(p, q);
		s.setPQ(p1, q1, 1);
		if(dis)
			s.setDisorder(dis);
		switch(rule)
		{
			case 0: s.mcs(n); break;
			case 1: s.mcsPQSyncRng(n); break;
			case 2: s.mcsDisorder2SyncRng(n); break;
			default: s.mcsEW(n);
		}
		s.popSystem(lat);
		s.getStreams(states);
		return 0;
	}
	catch(const std::exception& e)
	{
		std::fprintf(stderr, "%s\n", e.what());
		return -1;
	}
}
