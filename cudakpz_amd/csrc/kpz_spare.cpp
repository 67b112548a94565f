#include "kpz_spare.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <condition_variable>
#include <mutex>
#include <vector>

namespace kpz {

namespace {

// every SpareBuf of the process; one lock for all their state, held for a few
// instructions per use
struct Registry {
	std::mutex lock;
	std::condition_variable changed;
	std::vector<SpareBuf*> all;
};

// never destroyed: schedulers may outlive the library's static objects
Registry& registry()
{
	static Registry* const r = new Registry;
	return *r;
}

} // namespace

SpareBuf::SpareBuf()
{
	Registry& R = registry();
	std::lock_guard<std::mutex> hold(R.lock);
	R.all.push_back(this);
}

SpareBuf::~SpareBuf()
{
	Registry& R = registry();
	std::lock_guard<std::mutex> hold(R.lock);
	R.all.erase(std::find(R.all.begin(), R.all.end(), this));
	if(p_)
		(void)hipFree(p_);
	R.changed.notify_all();
}

void* SpareBuf::begin(size_t bytes, bool& fresh)
{
	Registry& R = registry();
	std::lock_guard<std::mutex> hold(R.lock);
	if(recalled_ || declined_)
		return nullptr;
	fresh = !p_;
	if(!p_)
	{
		// asked for once, and again after it was taken back
		declined_ = true;
		size_t free = 0, total = 0;
		if(hipGetDevice(&device_) != hipSuccess || hipMemGetInfo(&free, &total) != hipSuccess)
			return nullptr;
		size_t held = bytes;
		for(const SpareBuf* s : R.all)
			if(s->p_ && s->device_ == device_)
				held += s->n_;
		if(bytes > total / 64 || held > total / 16 || free < bytes || free - bytes < total / 4 * 3)
			return nullptr;
		if(hipMalloc(&p_, bytes) != hipSuccess)
		{
			(void)hipGetLastError();
			p_ = nullptr;
			return nullptr;
		}
		n_ = bytes;
		declined_ = false;
	}
	busy_ = true;
	return p_;
}

void SpareBuf::end()
{
	Registry& R = registry();
	std::lock_guard<std::mutex> hold(R.lock);
	busy_ = false;
	R.changed.notify_all();
}

uint64_t SpareBuf::takeBack(int device)
{
	Registry& R = registry();
	std::unique_lock<std::mutex> hold(R.lock);
	for(SpareBuf* s : R.all)
		if(s->p_ && s->device_ == device)
			s->recalled_ = true; // not used again before it is freed
	uint64_t freed = 0;
	for(;;)
	{
		SpareBuf* idle = nullptr;
		bool busy = false;
		for(SpareBuf* s : R.all)
			if(s->recalled_ && s->device_ == device)
			{
				if(s->busy_)
					busy = true;
				else
					idle = s;
			}
		if(idle)
		{
			(void)hipFree(idle->p_); // waits for the work queued on it
			idle->p_ = nullptr;
			idle->recalled_ = false;
			freed += idle->n_;
			R.changed.notify_all();
		}
		else if(busy)
			R.changed.wait(hold);
		else
			return freed;
	}
}

} // namespace kpz
