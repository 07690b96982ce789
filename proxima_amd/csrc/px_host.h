// px_host.h -- host-only helpers of libproxima_px.so (no HIP types).
#pragma once

#include <stdint.h>

#include <algorithm>
#include <thread>
#include <vector>

namespace px {

float host_l2_sqr(const float* a, const float* b, int64_t n);

// Host-side decisions of PQ training (pq.rs:54-95, 139-148): the training sample, and per
// subspace the initial centroids' sample rows [m][ks] and the generator state after them.
struct PqTrainPlan {
    int64_t n = 0, ks = 0;
    std::vector<int64_t> sample;
    std::vector<int64_t> init_rows;
    std::vector<uint64_t> rng_after_init;
};
void pq_train_plan(int64_t n_all, int64_t m, int64_t nbits, int64_t train_sample, uint64_t seed,
                   PqTrainPlan* plan);
void pq_gather_sample(const float* training, int64_t dim, int64_t m, const PqTrainPlan& plan,
                      float* out);
// The magnitude bits of the largest of len values (magnitudes order as their bits do):
// 0x7f800000 or more when one is NaN or infinite.
int32_t max_magnitude_bits(const float* x, int64_t len);
// Whether every value is exactly an fp16 zero or normal number: zero, or a magnitude in
// [2^-14, 2^16) with the 13 low mantissa bits clear -- what to_f16_kernel checks on the device.
bool f16_exact_values(const float* x, int64_t len);
// SplitMix64 below(n) (pq.rs:34-36) from *state, advancing it.
uint64_t splitmix_below(uint64_t* state, uint64_t n);
// Most roundings that a term of a key over n values passes in the reference's arithmetic
// (distance.rs:3-39): three of the squared difference (an inner product has one), its lane's
// sum over n / 8 chunks, the eight lanes' sum, and the n % 8 values added one by one.
inline int64_t ref_roundings(int64_t n) { return 3 + n / 8 + 8 + n % 8; }
// A screening scan's fp16 queries: values of all slots (a multiple of a wave's 64), and of the
// workgroup that its last fragment offsets may lie in, within 32-bit byte offsets.
constexpr int64_t kScreenBlockSlots = 512;
inline bool screen_batch_fits(int64_t nq, int64_t ds) {
    return ((nq + 63) / 64 * 64 + kScreenBlockSlots) * ds <= INT32_MAX / 2;
}
// The most queries (at most `most`) of ds padded dims that one screening scan takes; 0: none.
inline int64_t screen_batch(int64_t ds, int64_t most) {
    const int64_t slots = (INT32_MAX / 2 / ds - kScreenBlockSlots) / 64 * 64;
    return std::max<int64_t>(0, std::min(most, slots));
}
int host_threads();
// body(lo, hi) over [0, n) in one piece a host thread; where no more threads can be had, the
// calling one does the rest.
template <class F>
void parallel_for(int64_t n, F&& body) {
    const int nt = (int)std::min<int64_t>(host_threads(), std::max<int64_t>(n, 1));
    const int64_t per = (n + nt - 1) / nt;
    std::vector<std::thread> th;
    int64_t lo = per;
    try {
        th.reserve(nt);
        for (; lo < n; lo += per) {
            const int64_t hi = std::min(n, lo + per);
            th.emplace_back([&body, lo, hi] { body(lo, hi); });
        }
    } catch (...) {  // (no thread, or no memory for one)
    }
    body(0, std::min(per, n));
    if (lo < n) body(lo, n);
    for (auto& x : th) x.join();
}
void pq_train_host(const float* training, int64_t n_all, int64_t dim, int64_t m, int64_t nbits,
                   int64_t iters, int64_t train_sample, uint64_t seed, float* codebooks);
void pq_encode_host(const float* codebooks, int64_t dim, int64_t m, int64_t nbits,
                    const float* vectors, int64_t n, uint8_t* codes);

}  // namespace px
