// Test probe: parallel_for (gpu-smina_amd/host/parallel.h) under failing
// allocations and throwing bodies.  Arguments: n, grain, the first index that
// throws (-1: none), the allocation that fails (0: none), counted from the
// call.  Prints how the call ended and how often each index ran.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <stdexcept>
#include "../../gpu-smina_amd/host/parallel.h"

static std::atomic<long> left{0};
void* operator new(std::size_t n)
{
	if (left > 0 && --left == 0)
		throw std::bad_alloc();
	if (void* p = std::malloc(n ? n : 1))
		return p;
	throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

int main(int, char** a)
{
	const std::size_t n = std::size_t(std::atol(a[1]));
	const long bad = std::atol(a[3]);
	std::vector<std::atomic<int>> ran(n);
	const char* end = "done";
	char text[32];
	left = std::atol(a[4]);
	try
	{
		sgpu_host::parallel_for(n, std::size_t(std::atol(a[2])), [&](std::size_t i) {
			ran[i]++;
			if (bad >= 0 && long(i) >= bad)
				throw i;
		});
	}
	catch (std::size_t i)
	{
		std::snprintf(text, sizeof text, "threw %zu", i);
		end = text;
	}
	catch (std::bad_alloc&)
	{
		end = "bad_alloc";
	}
	left = 0;
	int lo = 1 << 30, hi = 0;
	for (auto& r : ran)
	{
		lo = std::min(lo, int(r));
		hi = std::max(hi, int(r));
	}
	std::printf("%s %d %d\n", end, n ? lo : 1, n ? hi : 1);
}
