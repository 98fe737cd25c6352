// Plans by circuit structure (host).  A program evaluates one structure many times with new gates; a
// plan costs from 20 us (6 qubits, 3 layers) to 0.8 ms (14 qubits, 9 layers).  The last kMost plans are
// kept (host memory only, given back by clear), fewer of large circuits: a gate takes 2 integers of the
// key and up to 1 KB of a plan, so that kMostInts bounds a cache at about 32 MB.  The key holds the
// whole structure, nothing of the gates.
#pragma once

#include <cstddef>
#include <functional>
#include <list>
#include <memory>
#include <mutex>
#include <utility>
#include <vector>

namespace rqc {

template <typename P>
class PlanCache
{
public:
	// Plans are made outside the lock, so that a thread with a new structure does not keep others from
	// theirs; of two threads that make the same plan the first one's is kept.
	std::shared_ptr<const P> get(const std::vector<int>& key, const std::function<std::shared_ptr<const P>()>& make)
	{
		if (auto p = find(key)) { return p; }
		auto made = make();
		std::lock_guard<std::mutex> lk(mu_);
		if (auto p = find_locked(key)) { return p; }
		plans_.emplace_front(key, made);
		ints_ += key.size();
		while (plans_.size() > 1 && (plans_.size() > kMost || ints_ > kMostInts)) {
			ints_ -= plans_.back().first.size();
			plans_.pop_back();
		}
		return made;
	}

	// (plans in use stay with their users)
	void clear()
	{
		std::lock_guard<std::mutex> lk(mu_);
		plans_.clear();
		ints_ = 0;
	}

private:
	static constexpr size_t kMost = 64, kMostInts = (size_t)1 << 16;
	std::mutex mu_;
	size_t ints_ = 0;   // of the keys kept
	std::list<std::pair<std::vector<int>, std::shared_ptr<const P>>> plans_;

	std::shared_ptr<const P> find(const std::vector<int>& key)
	{
		std::lock_guard<std::mutex> lk(mu_);
		return find_locked(key);
	}
	std::shared_ptr<const P> find_locked(const std::vector<int>& key)
	{
		for (auto it = plans_.begin(); it != plans_.end(); ++it) {
			if (it->first == key) {
				plans_.splice(plans_.begin(), plans_, it);
				return it->second;
			}
		}
		return nullptr;
	}
};

}  // namespace rqc
