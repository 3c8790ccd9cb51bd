// Device memory that a model holds between calls: what it cannot do without, and what it is faster with.  The allocator is the
// caller's, so that tests/cpp/fetch_bounds_test.cpp can refuse on the host what a card seldom does.
#pragma once

#include <cstddef>

namespace litenn_hip
{
	struct Room
	{
		void* data = nullptr;
		size_t bytes = 0;
		size_t refused = static_cast<size_t>(-1); // so much could not be had
	};

	// Makes the room hold `want` bytes (a size that was refused is not asked for again), or `need`, the lesser, where those cannot be had.
	// False: not even these, and the room is empty.  allocate(bytes): memory or null; release(memory): what it was may be used no more.
	template <typename Allocate, typename Release>
	bool grow_room(Room& room, size_t need, size_t want, Allocate&& allocate, Release&& release)
	{
		const size_t aim = want < room.refused ? want : need;
		if (room.data && room.bytes >= aim)
		{
			return true;
		}
		if (room.data)
		{
			release(room.data);
			room.data = nullptr;
			room.bytes = 0;
		}
		room.data = allocate(aim);
		room.bytes = room.data ? aim : 0;
		if (!room.data && aim > need)
		{
			room.refused = aim;
			room.data = allocate(need);
			room.bytes = room.data ? need : 0;
		}
		return room.data != nullptr;
	}
} // namespace litenn_hip
