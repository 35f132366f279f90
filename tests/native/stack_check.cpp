/*
 * The traversal stack (luxcore_amd/csrc/lrh_stack.h) against a plain one: a
 * ray's entries pushed and popped singly, then by a group of W lanes that push
 * up to W at a time, with the ring and the spill array between guard words and
 * other lanes' columns.  Pops give the plain stack's entries, a push reports
 * exactly where the entries pass the two arrays (a single one is refused,
 * after a shared one the ray goes on for a while with what there is), and
 * no word outside the ray's column changes.
 *
 *   stack_check <ldsDepth> <spillDepth> <W> <seed> <steps>
 * Prints "ok <pushes beyond> <deepest>" or what went wrong.
 */
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "../../luxcore_amd/csrc/lrh_stack.h"

namespace {

struct Entry {
	uint32_t x, y;
};

constexpr uint32_t kShift = 6, kLanes = 1u << kShift, kGuard = 0xdeadbeefu;

// rows x columns of entries with a row of guards before and after
struct Guarded {
	std::vector<Entry> v;
	uint32_t rows, cols, col;
	Guarded(uint32_t r, uint32_t c, uint32_t mine) : v((size_t)(r + 2) * c, Entry{kGuard, kGuard}), rows(r), cols(c), col(mine) {}
	Entry *data() { return v.data() + cols; }
	bool intact() const {
		for (size_t i = 0; i < v.size(); ++i) {
			const size_t row = i / cols;
			if (row >= 1 && row <= rows && i % cols == col) continue;
			if (v[i].x != kGuard || v[i].y != kGuard) return false;
		}
		return true;
	}
};

}  // namespace

int main(int argc, char **argv) {
	if (argc != 6) return 2;
	const uint32_t depth = (uint32_t)std::atoi(argv[1]), spillDepth = (uint32_t)std::atoi(argv[2]),
				   W = (uint32_t)std::atoi(argv[3]), steps = (uint32_t)std::atoi(argv[5]);
	std::mt19937 rng((uint32_t)std::atoi(argv[4]));
	const uint32_t lane = rng() % kLanes, glane0 = kLanes, gstride = 3 * kLanes;
	Guarded lds(depth, kLanes, lane), spill(spillDepth, gstride, glane0 + lane);
	lrhstack::Stack<Entry> s{lds.data(), spill.data(), kShift, lane, gstride, glane0, depth - 1, depth, spillDepth, 0};
	std::vector<uint32_t> plain;
	uint32_t next = 1, refused = 0, deepest = 0;
	auto bad = [&](const char *what, uint32_t step) {
		std::printf("%s at step %u, %u entries\n", what, step, (uint32_t)plain.size());
		std::exit(1);
	};
	for (uint32_t step = 0; step < steps; ++step) {
		const bool shared = step >= steps / 3;
		// runs of mostly pushes and of mostly pops
		const bool pushing = rng() % 8u < ((step / 64u) % 2u ? 2u : 6u);
		if (pushing && !shared) {
			bool full = false;
			const bool ok = lrhstack::push(s, Entry{next, ~next}, [&]() { full = true; });
			if (ok == full || ok != (plain.size() < depth + spillDepth)) bad("push", step);
			if (ok) plain.push_back(next++);
			else ++refused;
		} else if (pushing) {
			const uint32_t n = rng() % (W + 1u);
			bool full = false;
			// (the lanes' order does not matter: each has places of its own)
			const uint32_t from = n ? rng() % n : 0u;
			for (uint32_t k = 0; k < W; ++k) {
				const uint32_t i = n ? (from + k) % n : 0u;
				lrhstack::drainPush(s, k < n, s.sp + i, s.sp + n, Entry{next + i, ~(next + i)}, [&]() { full = true; });
			}
			s.sp += n;
			for (uint32_t i = 0; i < n; ++i) plain.push_back(next++);
			const bool over = plain.size() > depth + spillDepth;
			if (full != over || lrhstack::overfull(s) != over) bad("shared push", step);
			if (over) {
				// the ray goes on with what there is until it is ended
				++refused;
				for (uint32_t k = rng() % 300u; k > 0 && s.sp > 0; --k) {
					if (rng() % 3u) {
						if (lrhstack::drainPop(s, true).x == kGuard) bad("a word from outside the arrays", step);
					} else {
						const uint32_t m = rng() % (W + 1u);
						for (uint32_t i = 0; i < m; ++i)
							lrhstack::drainPush(s, true, s.sp + i, s.sp + m, Entry{next, ~next}, [&]() { full = true; });
						s.sp += m;
					}
				}
				s.sp = 0;
				plain.clear();
			}
		} else if (!plain.empty()) {
			Entry e;
			if (shared) {
				// every lane reads the top, the leader refills the ring
				lrhstack::Stack<Entry> other = s;
				const Entry seen = lrhstack::drainPop(other, false);
				e = lrhstack::drainPop(s, true);
				if (seen.x != e.x || other.sp != s.sp) bad("a follower's pop", step);
			} else
				e = lrhstack::pop(s);
			if (e.x != plain.back() || e.y != ~plain.back()) bad("pop", step);
			plain.pop_back();
		}
		if (s.sp != plain.size()) bad("depth", step);
		if (plain.size() > deepest) deepest = (uint32_t)plain.size();
		if (!lds.intact() || !spill.intact()) bad("a word outside the ray's column", step);
	}
	std::printf("ok %u %u\n", refused, deepest);
	return 0;
}
