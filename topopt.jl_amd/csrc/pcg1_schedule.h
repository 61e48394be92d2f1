// Which captured graphs of one-launch PCG iterations (k_pcg1.h) the host launches
// between two looks at the device's state.  Launches that find the solve done cost
// 1.3 to 2.5 us each, a look 15 to 20 us with the graph's start.
//
// First a graph of 32: solves from a near guess end in it (one of 64 took 366 against
// 258 us for an EnergyCriteria solve that stops at once, with its three kernels an
// iteration, and 294 against 242 us for an assembled one, MI355X).  Then graphs of
// 64, several per look while the residual's history or the iteration limit says that
// many are to go, and near the end shorter ones.
#pragma once
#include <algorithm>
#include <cmath>

namespace tohip {

enum { kPcg1Start, kPcg1Long, kPcg1Short, kPcg1Graphs };
// Even, so that a graph starts and ends on the first set of vectors.
constexpr int kPcg1GraphIters[kPcg1Graphs] = {32, 64, 8};

struct Pcg1Schedule {
    int graph = kPcg1Start, launches = 1;
    double prev_res = -1.0;
    long long prev_it = 0;

    // After `iter` iterations that did not end the solve, at r.r = rr (rr0 at the start).
    void next(long long iter, long long maxiter, double rr, double rr0, double tol) {
        const double res = std::sqrt(rr);
        const bool first = prev_res < 0;
        if (first) prev_res = std::sqrt(rr0);
        double togo = -1.0;
        if (prev_res > 0 && res > 0 && tol > 0 && iter > prev_it) {
            const double rate = std::log(res / prev_res) / double(iter - prev_it);
            if (rate < 0) togo = std::min(std::log(tol / res) / rate, 1e6);
        }
        prev_res = res;
        prev_it = iter;
        const double left = double(maxiter - iter);
        graph = kPcg1Long;
        launches = 1;
        if (togo < 0 && left >= 0.75 * kPcg1GraphIters[kPcg1Long]) return;  // no prediction
        togo = togo < 0 ? left : std::min(togo, left);
        if (togo >= 0.75 * kPcg1GraphIters[kPcg1Long]) {
            // (the first iterations say little about the rate to come)
            const int most = first ? 1 : 4;
            launches =
                std::max(1, std::min(most, (int)(togo / (1.5 * kPcg1GraphIters[kPcg1Long]))));
        } else if (togo >= 0.75 * kPcg1GraphIters[kPcg1Start]) {
            graph = kPcg1Start;
        } else {
            graph = kPcg1Short;
            launches = std::max(1, (int)(togo / kPcg1GraphIters[kPcg1Short]));
        }
    }
};

}  // namespace tohip
