// Device memory that only makes calls faster, held by its owner until something
// else needs the room.
#pragma once

#include <cstddef>
#include <cstdint>

namespace kpz {

// A buffer that may be taken back whenever its owner is not queueing work on it
// (hipFree waits for queued work).  A failing DevBuf::alloc takes back all those
// of its device and tries again; allocations that the library does not see
// (another library's, another process's) find the room after kpz_release_spares.
// So that these seldom need to, a buffer takes at most a 64th of the device's
// memory, all of a process's at most a 16th, and each is taken only while three
// quarters of the memory stay free after it.
class SpareBuf {
public:
	SpareBuf();
	~SpareBuf();
	SpareBuf(const SpareBuf&) = delete;
	SpareBuf& operator=(const SpareBuf&) = delete;

	// The buffer while work is queued on it.  Between the two ends nothing may
	// be allocated with DevBuf: it might wait for this buffer.
	class Use {
	public:
		Use(SpareBuf& b, size_t bytes) : b_(b), p_(b.begin(bytes, fresh_)) {}
		~Use()
		{
			if(p_)
				b_.end();
		}
		Use(const Use&) = delete;
		Use& operator=(const Use&) = delete;
		void* get() const { return p_; }      // null: not to be had
		bool fresh() const { return fresh_; } // nothing of an earlier use is in it

	private:
		SpareBuf& b_;
		bool fresh_ = false;
		void* p_;
	};

	// takes back all buffers on the device; bytes freed
	static uint64_t takeBack(int device);

private:
	void* begin(size_t bytes, bool& fresh);
	void end();
	void* p_ = nullptr;
	size_t n_ = 0;
	int device_ = -1;
	bool busy_ = false, recalled_ = false, declined_ = false;
};

} // namespace kpz
