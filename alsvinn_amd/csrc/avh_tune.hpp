// Tile shapes the autotuner chose, shared by every solver of the process.
//
// A choice holds for what was timed: the launches of one integrator's step on
// one equation, reconstruction, flux and grid.  The integrators' launches
// differ (RK3's last two stages are one launch on some shapes, RK2 forms its
// input as it loads, forward euler has one stage), and so do their best shapes.
#pragma once
#include <map>
#include <mutex>
#include <tuple>

#include "../../include/alsvinn_hip.h"

namespace avh {

enum TuneKind { TUNE_SOLVER = 0, TUNE_BATCH = 1 };
typedef std::tuple<int, int, int, int, int, int, long long, long long, long long> TuneKey;

// n: a solver's grid; of a batch the first group's nx and ny and its samples
inline TuneKey tune_key(TuneKind kind, const avh_config& c, int dim, const long long (&n)[3]) {
    return TuneKey(kind, c.equation, c.reconstruction, c.flux, c.integrator, dim, n[0], n[1], n[2]);
}

inline std::mutex& tune_mutex() {
    static std::mutex m;
    return m;
}

inline std::map<TuneKey, int>& tune_cache() {
    static std::map<TuneKey, int> c;
    return c;
}

inline bool tune_lookup(const TuneKey& k, int* shape) {
    std::lock_guard<std::mutex> g(tune_mutex());
    auto it = tune_cache().find(k);
    if (it == tune_cache().end()) return false;
    *shape = it->second;
    return true;
}

// `whole_step`: the step's launches were timed.  A solver that has stopped is
// timed on its first stage alone, which says nothing about the others': the
// choice is then its own.
inline void tune_store(const TuneKey& k, int shape, bool whole_step) {
    if (!whole_step) return;
    std::lock_guard<std::mutex> g(tune_mutex());
    tune_cache()[k] = shape;
}

}  // namespace avh
