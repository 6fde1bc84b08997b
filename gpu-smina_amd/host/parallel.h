/*
 * The host's loops over the ligands and chains of a batch, on threads.
 */
#ifndef SGPU_PARALLEL_H
#define SGPU_PARALLEL_H

#include <algorithm>
#include <cstddef>
#include <exception>
#include <thread>
#include <vector>

namespace sgpu_host
{

// f(0) .. f(n - 1) on up to 16 threads (one for small n), in runs of
// neighbouring indices; the exception of the lowest index that throws is
// rethrown
template<typename F>
void parallel_for(std::size_t n, std::size_t grain, F&& f)
{
	const std::size_t hw = std::max(1u, std::thread::hardware_concurrency());
	const std::size_t nt = std::min({std::size_t(16), hw, n / std::max<std::size_t>(1, grain)});
	if (nt < 2)
	{
		for (std::size_t i = 0; i < n; i++)
			f(i);
		return;
	}
	std::vector<std::exception_ptr> failed(nt);
	auto part = [&](std::size_t t) {
		try
		{
			for (std::size_t i = n * t / nt; i < n * (t + 1) / nt; i++)
				f(i);
		}
		catch (...)
		{
			failed[t] = std::current_exception();
		}
	};
	std::vector<std::thread> threads;
	threads.reserve(nt - 1); // (growing past a failure would end the process: threads run)
	std::size_t started = 1;
	try
	{
		for (; started < nt; started++)
			threads.emplace_back(part, started);
	}
	catch (...)
	{
		// no more threads, or no memory for one: this thread takes the parts
		// that have none
	}
	part(0);
	for (std::size_t t = started; t < nt; t++)
		part(t);
	for (std::thread& t : threads)
		t.join();
	for (const std::exception_ptr& e : failed)
		if (e)
			std::rethrow_exception(e);
}

} // namespace sgpu_host

#endif
