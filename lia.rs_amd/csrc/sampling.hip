// Sparse sampling after the paged step (gfx950): the candidates kernel and the host-side
// sampler of Engine::forward_paged_sampled (src/inference/paged_sampling.rs:7-76).
//
// The kernel (llama_nucleus_candidates, src/gpu/kernels/llama_nucleus.rs:18-117) gives one
// wavefront to each (row, part of 1024 vocabulary entries), whose load instructions read 1 KB
// each.  It writes the part's 21 largest entries by the total order of their f32 bits (ties: larger
// id first) as (id << 32 | bits) words, then the part's maximum and the f64 softmax mass
// sum exp((x - max) / T) (NaN when the part holds a NaN or +inf).  The host reduces the
// parts to one candidate list per row (src/gpu/nucleus.rs:103-143) and samples it: top-k
// from the candidates, nucleus only when the candidates prove the cutoff
// (checked_nucleus), else from the full logit row read back from the device.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "common.hpp"
#include "launch.hpp"

// Every product and sum below is rounded on its own, as in the reference (no FMA contraction).
#pragma clang fp contract(off)

namespace lia {

constexpr uint32_t kSlots = 21;   // 20 candidates + the omitted-tail bound (nucleus.rs:4)
constexpr uint32_t kPart = 1024;
constexpr uint32_t kPerLane = kPart / 64;

// f32::total_cmp as a signed key: negative values have their magnitude bits flipped.
__host__ __device__ __forceinline__ int32_t total_key(uint32_t bits) {
    const int32_t s = (int32_t)bits;
    return s ^ (int32_t)((uint32_t)(s >> 31) >> 1);
}

__device__ __forceinline__ bool better(int32_t key, uint32_t id, int32_t bkey, uint32_t bid) {
    return key > bkey || (key == bkey && id > bid);
}

// Number of (lane, j) entries of the wave with pred(j) true: one ballot and one scalar bit
// count per register.
template <typename Pred>
__device__ __forceinline__ uint32_t wave_count(Pred pred) {
    uint32_t n = 0;
#pragma unroll
    for (uint32_t j = 0; j < kPerLane; j++) n += __builtin_popcountll(__ballot(pred(j)));
    return n;
}

// One wavefront per (row, part).  The k = min(21, visible) best entries are found without
// k serial argmax rounds (keys biased to unsigned: u = key ^ 0x80000000):
//  - a tau that 21 lane maxima reach is a lower bound of the 21st largest entry (those maxima
//    are 21 distinct entries), so the entries >= tau - usually a few
//    dozen - contain the answer: when at most 64 survive they are ranked directly;
//  - otherwise (mass ties) a bit-by-bit search with ballot counts finds the k-th largest key
//    T, and a second search over the in-part offset settles ties at T (larger ids first).
// The selected entries are compacted into LDS and each lands at its rank.  "Visible" entries are the reference's selectable ones:
// inside the vocabulary and with a key above INT32_MIN (an all-ones NaN is never taken by
// its rounds).  Slots past k hold the reference's empty word (0xFFFFFFFF id, -inf bits).
__global__ __launch_bounds__(256) void nucleus_candidates_kernel(
        uint32_t vocab, uint32_t parts, uint32_t groups, const double *__restrict__ temperatures,
        const float *__restrict__ logits, uint64_t *__restrict__ candidates,
        double *__restrict__ normalizers) {
    __shared__ uint64_t stage[4][64];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t group = blockIdx.x * 4 + wave;
    if (group >= groups) return;                       // whole waves leave together
    const uint32_t row = group / parts, part = group % parts;
    const uint32_t base = part * kPart;
    const uint32_t live = min(vocab - base, kPart);
    // Bounded loads: entries past the part's live range read as 0 without touching memory,
    // so the loads are issued back to back with no branch.  Register j holds entry
    // 256 (j / 4) + 4 lane + j % 4 of the part: 16 bytes a lane and load.
    const auto rsrc = make_rsrc(logits + (size_t)row * vocab + base, live * 4);
    auto entry = [&](uint32_t j) { return 256 * (j / 4) + 4 * lane + j % 4; };
    float v[kPerLane];
#pragma unroll
    for (uint32_t j = 0; j < kPerLane; j += 4) {
        const f32x4 x = __builtin_bit_cast(f32x4, buffer_load16(rsrc, entry(j) * 4));
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) v[j + i] = x[i];
    }
    // Biased order keys u (0 = not visible), and from their extremes what most parts need: the
    // maximum, that no entry is NaN or +inf, that every entry is visible.  Keys order -inf above the
    // negative NaNs and +inf below the positive ones.
    constexpr uint32_t kNegInf = 0x007fffffu, kPosInf = 0xff800000u;
    uint32_t u[kPerLane], hi = 0, least = 0xffffffffu;
#pragma unroll
    for (uint32_t j = 0; j < kPerLane; j++) {
        const uint32_t s = __float_as_uint(v[j]);
        u[j] = s ^ ((uint32_t)((int32_t)s >> 31) | 0x80000000u);
        if (live < kPart && entry(j) >= live) u[j] = 0; // (live is uniform)
        hi = max(hi, u[j]);
        least = min(least, u[j]);
    }
    float mx = -INFINITY;
    bool invalid = false;
    const bool ordinary = !__any(hi >= kPosInf || least < kNegInf); // the whole part, no NaN, no +inf
    if (ordinary) {
        mx = __uint_as_float((uint32_t)total_key(hi ^ 0x80000000u));
    } else {
#pragma unroll
        for (uint32_t j = 0; j < kPerLane; j++) {
            const bool in = entry(j) < live;
            v[j] = in ? v[j] : -INFINITY;
            mx = fmaxf(mx, v[j]);                       // ignores NaN, as f32::max does
            invalid |= in && ((v[j] != v[j]) || v[j] == INFINITY);
        }
    }
#pragma unroll
    for (int o = 32; o; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    double sum = 0.0;
    const double t = temperatures[row];
    if (t > 0.0 && isfinite(mx)) {
        // Quotients by the row's temperature from its reciprocal, corrected by a fused remainder
        // (Markstein, "Computation of elementary functions on the IBM RISC System/6000", 1990): five
        // operations, where the division sequence takes eleven.  Both sides are scaled to a
        // temperature in [0.5, 1), and quotients below -1e6 (whose exponential is 0) cut, so no
        // step leaves the exponent range.  An infinite temperature gives the weights of the largest
        // finite one, 1 each.
        int e2;
        const double ts = __builtin_frexp(fmin(t, 0x1.fffffffffffffp1023), &e2), inv = 1.0 / ts;
#pragma unroll
        for (uint32_t j = 0; j < kPerLane; j++) {
            const double x = fmax(__builtin_ldexp((double)v[j] - (double)mx, -e2), -1e6);
            const double q = x * inv;
            const double e = exp(__builtin_fma(__builtin_fma(-q, ts, x), inv, q));
            sum += isfinite(v[j]) ? e : 0.0;
        }
    }
    if (__any(invalid)) sum = NAN;
#pragma unroll
    for (int o = 32; o; o >>= 1) sum += __shfl_xor(sum, o);
    if (lane == 0) {
        normalizers[2 * (size_t)group] = (double)mx;
        normalizers[2 * (size_t)group + 1] = sum;
    }

    const uint32_t visible = ordinary ? kPart : wave_count([&](uint32_t j) { return u[j] != 0; });
    const uint32_t k = min(visible, kSlots);
    // selection: u >= lo, and at u == lo only offsets >= I
    uint32_t lo = 1, I = 0, n_sel = k;
    if (k == kSlots) {
        // a bound that at least 21 lane maxima reach, and at most a few more
        uint32_t tau = 0;
        for (int bit = 31; bit >= 0; bit--) {
            const uint32_t c = tau | (1u << bit);
            const uint32_t n = (uint32_t)__builtin_popcountll(__ballot(hi >= c));
            if (n >= kSlots) tau = c;
            if (n >= kSlots && n <= kSlots + 4) break;
        }
        const uint32_t n_s = tau ? wave_count([&](uint32_t j) { return u[j] >= tau; }) : 1024u;
        if (n_s <= 64) {
            lo = tau;
            n_sel = n_s;
        } else {
            uint32_t T = 0;                             // largest T with count(u >= T) >= 21
            for (int bit = 31; bit >= 0; bit--) {
                const uint32_t c = T | (1u << bit);
                if (wave_count([&](uint32_t j) { return u[j] >= c; }) >= kSlots) T = c;
            }
            const uint32_t r = kSlots - wave_count([&](uint32_t j) { return u[j] > T; });
            for (int bit = 9; bit >= 0; bit--) {        // the r largest offsets among u == T
                const uint32_t c = I | (1u << bit);
                if (wave_count([&](uint32_t j) { return u[j] == T && entry(j) >= c; }) >= r) I = c;
            }
            lo = T;
        }
    }
    // compact the n_sel selected entries into LDS (any order), then rank them: key << 32 | offset
    // orders them, slots past n_sel hold 0 and rank below, so the reads go out eight at a time
    stage[wave][lane] = 0;
    uint32_t at = 0;
#pragma unroll
    for (uint32_t j = 0; j < kPerLane; j++) {
        const uint32_t off = entry(j);
        const bool sel = k && (u[j] > lo || (u[j] == lo && off >= I));
        const uint64_t m = __ballot(sel);
        if (sel) {
            const uint32_t pos = at + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                               __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
            stage[wave][pos] = (uint64_t)u[j] << 32 | off;
        }
        at += __builtin_popcountll(m);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    uint64_t word = (uint64_t)0xFFFFFFFFu << 32 | __float_as_uint(-INFINITY);
    uint32_t rank = lane;                               // lanes k..20: empty slots
    if (lane < n_sel) {
        const uint64_t mine = stage[wave][lane];
        rank = 0;
        for (uint32_t m = 0; m < n_sel; m += 8) {
#pragma unroll
            for (uint32_t i = 0; i < 8; i++) rank += stage[wave][m + i] > mine;
        }
        const uint32_t bits = (uint32_t)total_key((uint32_t)(mine >> 32) ^ 0x80000000u); // the key map is an involution
        word = (uint64_t)(base + (uint32_t)mine) << 32 | bits;
    }
    if (rank < kSlots) candidates[(size_t)group * kSlots + rank] = word;
}

// One row's parts reduced for the host: the sums over its parts and its kRowWords best candidates
// (ranks 0 .. 19 of every part) by the candidate order.  kept = 0 with candidates there means that
// too many tie for a place; the host then reads the row's part records.
constexpr uint32_t kRowWords = 128;   // select_nucleus's first prefix
struct RowSummary {
    double maximum, total;            // over the parts; total: the softmax mass at `maximum`
    float omitted;                    // largest candidate left out of a part's 20
    uint32_t kept, count;             // words below, candidates in all
    uint32_t invalid;                 // some part's mass is not finite
    uint64_t words[kRowWords];        // (id << 32 | f32 bits), best first
};

constexpr uint32_t kRowThreads = 512, kRowStage = 256;

// One workgroup per row; W words of the row's records per thread.  The host's reduction reads 21
// words of each of a row's parts (23.5 KB a row at 130,560 entries) and sorts 2,560 candidates: 64
// rows took 27 us to copy and about 600 us of one host core.  Here: a bit-by-bit search with ballot
// counts for a threshold that 128 to 256 candidates pass (one barrier a step, and it stops at the
// first such threshold), then each survivor's rank among the survivors.  Bound by the search's
// barriers and the loads before it (10.6 us for 64 rows); the copy is 1,056 bytes a row.
template <int W>
__global__ __launch_bounds__(kRowThreads) void nucleus_rows_kernel(
        uint32_t parts, const double *__restrict__ temperatures, const uint64_t *__restrict__ candidates,
        const double *__restrict__ normalizers, RowSummary *__restrict__ summaries) {
    constexpr uint32_t WAVES = kRowThreads / 64;
    __shared__ uint64_t s_key[kRowStage];
    __shared__ uint32_t s_cnt[2][WAVES], s_omit[WAVES], s_bad[WAVES], s_n;
    __shared__ double s_max[WAVES], s_sum[WAVES];
    const uint32_t row = blockIdx.x, t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const uint64_t *words = candidates + (size_t)row * parts * kSlots;
    const uint32_t n_words = parts * kSlots;
    RowSummary *out = summaries + row;
    if (t == 0) s_n = 0;
    uint32_t u[W], id[W], omit = 0;   // biased order keys of the finite values, 0 = none
#pragma unroll
    for (int c = 0; c < W; c++) {
        const uint32_t i = c * kRowThreads + t;
        const uint64_t w = words[min(i, n_words - 1)];
        const uint32_t bits = (uint32_t)w;
        id[c] = (uint32_t)(w >> 32);
        const bool live = i < n_words && id[c] != 0xFFFFFFFFu && (bits & 0x7f800000u) != 0x7f800000u;
        const uint32_t key = live ? (uint32_t)total_key(bits) ^ 0x80000000u : 0u;
        const bool last = i % kSlots == kSlots - 1;
        u[c] = last ? 0u : key;
        omit = max(omit, last ? key : 0u);
    }
    double mx = -INFINITY, mass = 0.0;
    bool bad = false;
    if (t < parts) {
        const double *ns = normalizers + ((size_t)row * parts + t) * 2;
        mx = ns[0];
        mass = ns[1];
        bad = !isfinite(mass);
    }
    double m = mx;
#pragma unroll
    for (int o = 32; o; o >>= 1) {
        m = fmax(m, __shfl_xor(m, o));
        omit = max(omit, (uint32_t)__shfl_xor((int)omit, o));
    }
    const bool any_bad = __any(bad);
    if (lane == 0) {
        s_max[wave] = m;
        s_omit[wave] = omit;
        s_bad[wave] = any_bad;
    }
    // candidates with keys >= bound, over the workgroup
    uint32_t turn = 0;
    auto count = [&](uint32_t bound) {
        uint32_t n = 0;
#pragma unroll
        for (int c = 0; c < W; c++) n += __builtin_popcountll(__ballot(u[c] >= bound));
        if (lane == 0) s_cnt[turn][wave] = n;
        lds_barrier();
        n = 0;
#pragma unroll
        for (uint32_t w = 0; w < WAVES; w++) n += s_cnt[turn][w];
        turn ^= 1;
        return n;
    };
    const uint32_t all = count(1); // (also publishes the maxima)
    double maximum = -INFINITY;
#pragma unroll
    for (uint32_t w = 0; w < WAVES; w++) maximum = fmax(maximum, s_max[w]);
    const double temp = temperatures[row];
    double sum = t < parts && temp > 0.0 && mass > 0.0 ? mass * exp((mx - maximum) / temp) : 0.0;
#pragma unroll
    for (int o = 32; o; o >>= 1) sum += __shfl_xor(sum, o);
    if (lane == 0) s_sum[wave] = sum;
    uint32_t bound = 1, n = all;
    if (all > kRowStage) {
        bound = 0;
        for (int bit = 31; bit >= 0; bit--) { // the counts are the same in every thread
            const uint32_t b = bound | (1u << bit);
            const uint32_t k = count(b);
            if (k >= kRowWords) {
                bound = b;
                n = k;
                if (k <= kRowStage) break;
            }
        }
    }
    const bool fits = n <= kRowStage;
    if (fits) {
#pragma unroll
        for (int c = 0; c < W; c++)
            if (u[c] >= bound) s_key[atomicAdd(&s_n, 1u)] = (uint64_t)u[c] << 32 | id[c];
    }
    lds_barrier();
    if (fits && t < n) {
        const uint64_t mine = s_key[t];
        uint32_t rank = 0;
#pragma unroll 8
        for (uint32_t k = 0; k < n; k++) rank += s_key[k] > mine;
        if (rank < kRowWords)
            out->words[rank] = mine << 32 | (uint32_t)total_key((uint32_t)(mine >> 32) ^ 0x80000000u);
    }
    if (t == 0) {
        double total = 0.0;
        uint32_t om = 0, inv = 0;
#pragma unroll
        for (uint32_t w = 0; w < WAVES; w++) {
            total += s_sum[w];
            om = max(om, s_omit[w]);
            inv |= s_bad[w];
        }
        out->maximum = maximum;
        out->total = total;
        out->omitted = om ? __uint_as_float((uint32_t)total_key(om ^ 0x80000000u)) : -INFINITY;
        out->kept = fits ? min(n, kRowWords) : 0u;
        out->count = all;
        out->invalid = inv;
    }
}

// ------------------------------------------------------------------ host sampler

// MT19937 and the reference sampler's two-word canonical double (src/sampling/random.rs).
struct Mt19937 {
    uint32_t w[624];
    uint32_t index = 624;
    explicit Mt19937(uint32_t seed) {
        w[0] = seed;
        for (uint32_t i = 1; i < 624; i++) w[i] = 1812433253u * (w[i - 1] ^ (w[i - 1] >> 30)) + i;
    }
    uint32_t next() {
        if (index == 624) {
            for (uint32_t i = 0; i < 624; i++) {
                const uint32_t mixed = (w[i] & 0x80000000u) | (w[(i + 1) % 624] & 0x7fffffffu);
                w[i] = w[(i + 397) % 624] ^ (mixed >> 1) ^ ((mixed & 1) ? 0x9908b0dfu : 0u);
            }
            index = 0;
        }
        uint32_t v = w[index++];
        v ^= v >> 11;
        v ^= (v << 7) & 0x9d2c5680u;
        v ^= (v << 15) & 0xefc60000u;
        return v ^ (v >> 18);
    }
    double uniform() {
        const double low = next(), high = next();
        return std::min((low + high * 4294967296.0) / 18446744073709551616.0, std::nextafter(1.0, 0.0));
    }
};

// Position-keyed Gumbel-max draw (src/sampling/gumbel.rs): MurmurHash3 mixing of
// (seed lo, seed hi, position lo, token), a 32-bit uniform, and -ln(-ln(1-u)) with a
// series for small u.
static uint32_t rotl(uint32_t x, int r) { return (x << r) | (x >> (32 - r)); }
static uint32_t gumbel_hash(uint64_t seed, uint64_t position, uint32_t token) {
    uint32_t h = 0;
    const uint32_t words[4] = {(uint32_t)seed, (uint32_t)(seed >> 32), (uint32_t)position, token};
    for (uint32_t word : words) {
        const uint32_t k = rotl(word * 0xcc9e2d51u, 15) * 0x1b873593u;
        h = rotl(h ^ k, 13) * 5u + 0xe6546b64u;
    }
    h ^= 16;
    h ^= h >> 16;
    h *= 0x85ebca6bu;
    h ^= h >> 13;
    h *= 0xc2b2ae35u;
    return h ^ (h >> 16);
}
static float gumbel_uniform(uint32_t word) {
    return (float)(word >> 16) * (1.0f / 65536.0f) + ((float)(word & 65535) + 0.5f) * (1.0f / 4294967296.0f);
}
static float gumbel_noise(float u) {
    float negative_log;
    if (u < 0.25f) {
        float poly = 1.0f / 8.0f;
        for (int d = 7; d >= 1; d--) poly = fmaf(u, poly, 1.0f / (float)d);
        negative_log = u * poly;
    } else {
        negative_log = -logf(std::max(1.0f - u, 1.0f / 16777216.0f));
    }
    return -logf(negative_log);
}

using Cand = std::pair<uint32_t, float>;   // (token id, logit)
using Entry = std::pair<uint32_t, double>; // (token id, probability)

static int32_t key_of(float x) {
    uint32_t b;
    memcpy(&b, &x, 4);
    return total_key(b);
}
// The reference's candidate order: descending total order of the logit, then descending id.
static bool before(const Cand &a, const Cand &b) {
    const int32_t ka = key_of(a.second), kb = key_of(b.second);
    return ka != kb ? ka > kb : a.first > b.first;
}

} // namespace lia

using namespace lia;

struct lia_sampler {
    double temperature, top_p;
    uint32_t top_k;
    uint64_t seed;
    bool keyed;
    uint64_t position;
    Mt19937 random;
    lia_sampler(double t, uint32_t k, double p, uint64_t s, bool keyed)
        : temperature(t), top_p(p), top_k(k), seed(s), keyed(keyed), position(0), random((uint32_t)s) {}

    double weight(float v, double maximum) const { return std::exp(((double)v - maximum) / temperature); }

    // Sampling::distribution (src/sampling.rs:82-128).
    int distribution(std::vector<Cand> c, std::vector<Entry> &out) const {
        for (const Cand &x : c)
            if (std::isnan(x.second) || x.second == INFINITY) return LIA_E_SAMPLING_LOGITS;
        c.erase(std::remove_if(c.begin(), c.end(), [](const Cand &x) { return x.second == -INFINITY; }),
                c.end());
        if (top_k && c.size() > top_k) {
            std::nth_element(c.begin(), c.begin() + top_k, c.end(), before);
            c.resize(top_k);
        }
        std::sort(c.begin(), c.end(), before);
        if (c.empty()) return LIA_E_EMPTY_DISTRIBUTION;
        {
            std::vector<uint32_t> ids(c.size());
            for (size_t i = 0; i < c.size(); i++) ids[i] = c[i].first;
            std::sort(ids.begin(), ids.end());
            if (std::adjacent_find(ids.begin(), ids.end()) != ids.end()) return LIA_E_DUPLICATE_CANDIDATE;
        }
        const double mx = c[0].second;
        out.resize(c.size());
        double total = 0.0;
        for (size_t i = 0; i < c.size(); i++) {
            out[i] = {c[i].first, std::exp(((double)c[i].second - mx) / temperature)};
        }
        for (const Entry &e : out) total += e.second;
        double mass = 0.0;
        size_t keep = out.size();
        for (size_t i = 0; i < out.size(); i++) {
            mass += out[i].second;
            if (mass >= top_p * total) {
                keep = i + 1;
                break;
            }
        }
        out.resize(keep);
        total = 0.0;
        for (const Entry &e : out) total += e.second;
        for (Entry &e : out) e.second /= total;
        return LIA_OK;
    }

    // select_nucleus (src/sampling/nucleus.rs:96-124); leaves c's retained prefix sorted.
    int select_nucleus(std::vector<Cand> &c, double maximum, double total, std::vector<Entry> &out) const {
        if (c.empty()) return LIA_E_EMPTY_DISTRIBUTION;
        const double target = top_p * total;
        size_t count = std::min<size_t>(c.size(), 128);
        for (;;) {
            if (count < c.size()) {
                std::nth_element(c.begin(), c.begin() + count, c.end(), before);
                std::sort(c.begin(), c.begin() + count, before);
            }
            double mass = 0.0;
            for (size_t i = 0; i < count; i++) mass += weight(c[i].second, maximum);
            if (mass >= target || count == c.size()) break;
            count = std::min(count * 2, c.size());
        }
        std::sort(c.begin(), c.begin() + count, before);
        double mass = 0.0;
        out.clear();
        for (size_t i = 0; i < count; i++) {
            const double w = weight(c[i].second, maximum);
            mass += w;
            out.push_back({c[i].first, w});
            if (mass >= target) break;
        }
        if (!std::isfinite(mass) || !(mass > 0.0)) return LIA_E_NUCLEUS;
        for (Entry &e : out) e.second /= mass;
        return LIA_OK;
    }

    // distribution_logits (nucleus.rs:9-46): the full-row fallback.
    int distribution_logits(const float *logits, uint32_t vocab, std::vector<Entry> &out) const {
        std::vector<Cand> c;
        c.reserve(vocab);
        if (top_k != 0 || top_p == 1.0) {
            for (uint32_t i = 0; i < vocab; i++) c.push_back({i, logits[i]});
            return distribution(std::move(c), out);
        }
        for (uint32_t i = 0; i < vocab; i++)
            if (std::isnan(logits[i]) || logits[i] == INFINITY) return LIA_E_SAMPLING_LOGITS;
        for (uint32_t i = 0; i < vocab; i++)
            if (logits[i] != -INFINITY) c.push_back({i, logits[i]});
        if (c.empty()) return LIA_E_EMPTY_DISTRIBUTION;
        float mx = c[0].second;
        for (const Cand &x : c)
            if (key_of(x.second) > key_of(mx)) mx = x.second;
        double total = 0.0;
        for (const Cand &x : c) total += weight(x.second, (double)mx);
        return select_nucleus(c, (double)mx, total, out);
    }

    // checked_nucleus (nucleus.rs:49-93): 1 with out set, 0 when the sparse candidates cannot
    // prove the cutoff (the caller falls back to the full row), or a negative status.
    int checked_nucleus(std::vector<Cand> c, double maximum, double total, float omitted,
                        std::vector<Entry> &out) const {
        if (!std::isfinite(total) || !(total > 0.0) || !std::isfinite(maximum)) return LIA_E_NUCLEUS;
        if (top_p == 1.0) return 0;
        const int st = select_nucleus(c, maximum, total, out);
        if (st) return st;
        if (out.empty()) return 0;
        const size_t keep = out.size();
        if (c[keep - 1].first != out.back().first) return LIA_E_NUCLEUS;
        if (!(key_of(c[keep - 1].second) > key_of(omitted))) return 0;
        const double target = top_p * total;
        double through = 0.0;
        for (size_t i = 0; i < keep; i++) through += weight(c[i].second, maximum);
        const double before_last = through - weight(c[keep - 1].second, maximum);
        const double uncertainty = std::fabs(total) * 1e-10;
        if (before_last >= target - uncertainty || through <= target + uncertainty) return 0;
        return 1;
    }

    // checked_nucleus on the `kept` best of `count` candidates, best first: the same sums in the same
    // order, taken only until the cutoff.  2: the cutoff lies past them.
    int checked_nucleus_best(const uint64_t *words, uint32_t kept, uint32_t count, double maximum,
                             double total, float omitted, std::vector<Entry> &out) const {
        if (!std::isfinite(total) || !(total > 0.0) || !std::isfinite(maximum)) return LIA_E_NUCLEUS;
        if (top_p == 1.0) return 0;
        if (kept == 0) return LIA_E_EMPTY_DISTRIBUTION;
        const double target = top_p * total;
        double mass = 0.0, w = 0.0;
        float last = 0.0f;
        out.clear();
        for (uint32_t i = 0; i < kept && !(i && mass >= target); i++) {
            const uint32_t bits = (uint32_t)words[i];
            memcpy(&last, &bits, 4);
            w = weight(last, maximum);
            mass += w;
            out.push_back({(uint32_t)(words[i] >> 32), w});
        }
        if (!(mass >= target) && kept < count) return 2;
        if (!std::isfinite(mass) || !(mass > 0.0)) return LIA_E_NUCLEUS;
        for (Entry &e : out) e.second /= mass;
        if (!(key_of(last) > key_of(omitted))) return 0;
        const double uncertainty = std::fabs(total) * 1e-10;
        return mass - w >= target - uncertainty || mass <= target + uncertainty ? 0 : 1;
    }

    // Sampling::draw (src/sampling.rs:134-146).
    uint32_t draw(const std::vector<Entry> &d) {
        if (keyed) {
            const uint64_t pos = position++;
            uint32_t best = d[0].first;
            float best_score = 0.0f;
            bool have = false;
            for (const Entry &e : d) {
                const float score = (float)std::log(e.second) + gumbel_noise(gumbel_uniform(gumbel_hash(seed, pos, e.first)));
                const int32_t k = key_of(score), bk = key_of(best_score);
                if (!have || k > bk || (k == bk && e.first < best)) {
                    best = e.first;
                    best_score = score;
                    have = true;
                }
            }
            return best;
        }
        if (d.size() == 1) return d[0].first;
        const double sample = random.uniform();
        double cumulative = 0.0;
        for (const Entry &e : d) {
            cumulative += e.second;
            if (sample < cumulative) return e.first;
        }
        return d.back().first;
    }
};

extern "C" int lia_sampler_create(double temperature, uint32_t top_k, double top_p, uint64_t seed,
                                  int32_t position_keyed, lia_sampler **out) {
    if (!out) return LIA_E_ARG;
    if (!std::isfinite(temperature) || !(temperature > 0.0) || top_k > 20 || !std::isfinite(top_p) ||
        !(top_p > 0.0) || top_p > 1.0)
        return LIA_E_SAMPLER_SETTINGS; // Sampling::new (src/sampling.rs:33-58)
    *out = new lia_sampler(temperature, top_k, top_p, seed, position_keyed != 0);
    return LIA_OK;
}

extern "C" void lia_sampler_destroy(lia_sampler *s) { delete s; }

extern "C" void lia_sampler_set_position(lia_sampler *s, uint64_t position) {
    if (s && s->keyed) s->position = position;
}

extern "C" int lia_sampler_distribution(const lia_sampler *s, uint32_t n, const uint32_t *ids,
                                        const float *logits, uint32_t *out_ids, double *out_probs,
                                        uint32_t *n_out) {
    if (!s || !n_out || (n && (!ids || !logits || !out_ids || !out_probs))) return LIA_E_ARG;
    std::vector<Cand> c(n);
    for (uint32_t i = 0; i < n; i++) c[i] = {ids[i], logits[i]};
    std::vector<Entry> d;
    const int st = s->distribution(std::move(c), d);
    if (st) return st;
    for (size_t i = 0; i < d.size(); i++) {
        out_ids[i] = d[i].first;
        out_probs[i] = d[i].second;
    }
    *n_out = (uint32_t)d.size();
    return LIA_OK;
}

extern "C" int lia_sampler_draw(lia_sampler *s, uint32_t n, const uint32_t *ids, const double *probs,
                                uint32_t *token) {
    if (!s || !token || n == 0 || !ids || !probs) return LIA_E_ARG;
    std::vector<Entry> d(n);
    for (uint32_t i = 0; i < n; i++) d[i] = {ids[i], probs[i]};
    *token = s->draw(d);
    return LIA_OK;
}

static uint32_t nucleus_parts(uint32_t vocab) { return (vocab + kPart - 1) / kPart; }
static size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

// Bytes of the part records and temperatures of `rows` rows.
static size_t record_bytes(uint32_t vocab, uint32_t rows) {
    const size_t g = (size_t)rows * nucleus_parts(vocab);
    return align_up(g * kSlots * 8, 256) + align_up(g * 16, 256) + align_up((size_t)rows * 8, 256);
}

// Rows whose records are reduced on the device: from 13 parts (more than two kRowWords lists: below,
// the records are about as small as the summary), up to the words the kernel's threads hold.
static bool summarised(uint32_t vocab) {
    const uint32_t words = nucleus_parts(vocab) * kSlots;
    return words > 2 * kRowWords && words <= 16 * kRowThreads;
}

extern "C" size_t lia_nucleus_workspace_bytes(uint32_t vocab, uint32_t rows) {
    return record_bytes(vocab, rows) + (summarised(vocab) ? (size_t)rows * sizeof(RowSummary) : 0);
}

extern "C" size_t lia_nucleus_host_bytes(uint32_t vocab, uint32_t rows) {
    return record_bytes(vocab, rows) + (size_t)vocab * 4;
}

extern "C" int lia_nucleus_candidates(uint32_t vocab, uint32_t rows, const double *temperatures,
                                      const float *logits, uint64_t *candidates,
                                      double *normalizers, lia_stream_t stream) {
    if (vocab == 0 || !temperatures || !logits || !candidates || !normalizers) return LIA_E_ARG;
    if (rows == 0) return LIA_OK;
    const uint64_t groups = (uint64_t)rows * nucleus_parts(vocab);
    if (groups > 0x3FFFFFFFu || (uint64_t)rows * vocab > 0xFFFFFFFFull) return LIA_E_ARG;
    const hipError_t e = launch<nucleus_candidates_kernel>(
        dim3((uint32_t)((groups + 3) / 4)), dim3(256), 0, (hipStream_t)stream, vocab,
        nucleus_parts(vocab), (uint32_t)groups, temperatures, logits, candidates, normalizers);
    return e == hipSuccess ? LIA_OK : LIA_E_HIP;
}

// A row's draw from its distribution, or by the sampler's fallback on its full logits (st = 0 of a
// nucleus row: `fetch(dst)` provides them).
template <typename Fetch>
static int finish_row(uint32_t vocab, lia_sampler *s, int st, std::vector<Entry> &d, std::vector<float> &row,
                      uint32_t *token, uint64_t *fallbacks, Fetch fetch) {
    if (st == 0 && s->top_k == 0) {
        if (fallbacks) ++*fallbacks;
        row.resize(vocab);
        st = fetch(row.data());
        if (st == LIA_OK) st = s->distribution_logits(row.data(), vocab, d);
    } else if (st == 1) {
        st = LIA_OK;
    }
    if (st) return st;
    *token = s->draw(d);
    return LIA_OK;
}

// Workspace::read's reduction of one row's part records and its sampling as forward_paged_sampled
// does it, on host records.
template <typename Fetch>
static int sample_parts(uint32_t vocab, lia_sampler *s, double temp, const uint64_t *cand, const double *ns,
                        std::vector<Cand> &c, std::vector<Entry> &d, std::vector<float> &row,
                        uint32_t *token, uint64_t *fallbacks, Fetch fetch) {
    const uint32_t parts = nucleus_parts(vocab);
    double maximum = -INFINITY;
    for (uint32_t p = 0; p < parts; p++) {
        if (!std::isfinite(ns[2 * p + 1])) return LIA_E_SAMPLING_LOGITS;
        if (ns[2 * p] > maximum) maximum = ns[2 * p];
    }
    double total = 0.0;
    if (temp > 0.0)
        for (uint32_t p = 0; p < parts; p++)
            if (ns[2 * p + 1] > 0.0) total += ns[2 * p + 1] * std::exp((ns[2 * p] - maximum) / temp);
    c.clear();
    float omitted = -INFINITY;
    for (uint32_t p = 0; p < parts; p++) {
        const uint64_t *words = cand + (size_t)p * kSlots;
        for (uint32_t rank = 0; rank < kSlots; rank++) {
            const uint32_t id = (uint32_t)(words[rank] >> 32);
            const uint32_t bits = (uint32_t)words[rank];
            float v;
            memcpy(&v, &bits, 4);
            if (id == 0xFFFFFFFFu || !std::isfinite(v)) continue;
            if (id >= vocab) return LIA_E_NUCLEUS;
            if (rank < kSlots - 1) c.push_back({id, v});
            else omitted = std::max(omitted, v);
        }
    }
    if (s) {
        const int st = s->top_k != 0 ? s->distribution(c, d) : s->checked_nucleus(c, maximum, total, omitted, d);
        return finish_row(vocab, s, st, d, row, token, fallbacks, fetch);
    }
    if (c.empty()) return LIA_E_EMPTY_DISTRIBUTION;
    Cand best = c[0];
    for (const Cand &x : c) {
        const int32_t k = key_of(x.second), bk = key_of(best.second);
        if (k > bk || (k == bk && x.first > best.first)) best = x;
    }
    *token = best.first;
    return LIA_OK;
}

// The same from the row's device summary.  2: it does not settle the row, the part records do.
template <typename Fetch>
static int sample_summary(uint32_t vocab, lia_sampler *s, const RowSummary &r, std::vector<Cand> &c,
                          std::vector<Entry> &d, std::vector<float> &row, uint32_t *token,
                          uint64_t *fallbacks, Fetch fetch) {
    if (r.invalid) return LIA_E_SAMPLING_LOGITS;
    if (r.kept == 0 && r.count) return 2;
    if (!s) {
        if (r.kept == 0) return LIA_E_EMPTY_DISTRIBUTION;
        *token = (uint32_t)(r.words[0] >> 32);
        return LIA_OK;
    }
    int st;
    if (s->top_k != 0) { // at most 20: the best of all candidates are among the best kRowWords
        c.clear();
        for (uint32_t i = 0; i < r.kept && i < s->top_k; i++) {
            const uint32_t bits = (uint32_t)r.words[i];
            float v;
            memcpy(&v, &bits, 4);
            c.push_back({(uint32_t)(r.words[i] >> 32), v});
        }
        st = s->distribution(c, d);
    } else {
        st = s->checked_nucleus_best(r.words, r.kept, r.count, r.maximum, r.total, r.omitted, d);
        if (st == 2) return 2;
    }
    return finish_row(vocab, s, st, d, row, token, fallbacks, fetch);
}

static void temperatures_for(uint32_t n, lia_sampler *const *samplers, double *t) {
    for (uint32_t i = 0; i < n; i++) {
        const lia_sampler *s = samplers ? samplers[i] : nullptr;
        t[i] = s ? (s->top_k == 0 ? s->temperature : 0.0) : 0.0;
    }
}

extern "C" int lia_sample_host(uint32_t vocab, uint32_t n, lia_sampler *const *samplers,
                               const uint32_t *positions, const uint64_t *candidates,
                               const double *normalizers, const float *logits, uint32_t *tokens,
                               uint64_t *fallbacks) {
    if (vocab == 0 || (n && (!candidates || !normalizers || !tokens))) return LIA_E_ARG;
    for (uint32_t i = 0; i < n; i++)
        if (samplers && samplers[i] && positions) lia_sampler_set_position(samplers[i], positions[i]);
    std::vector<double> t(n);
    temperatures_for(n, samplers, t.data());
    std::vector<Cand> c;
    std::vector<Entry> d;
    std::vector<float> row;
    const size_t parts = nucleus_parts(vocab);
    for (uint32_t r = 0; r < n; r++) {
        const int st = sample_parts(vocab, samplers ? samplers[r] : nullptr, t[r], candidates + r * parts * kSlots,
                                    normalizers + r * parts * 2, c, d, row, tokens + r, fallbacks, [&](float *dst) {
                                        if (!logits) return LIA_E_ARG;
                                        memcpy(dst, logits + (size_t)r * vocab, (size_t)vocab * 4);
                                        return LIA_OK;
                                    });
        if (st) return st;
    }
    return LIA_OK;
}

extern "C" int lia_sample_paged(uint32_t vocab, uint32_t n, lia_sampler *const *samplers,
                                const uint32_t *positions, const float *logits, void *workspace,
                                size_t workspace_bytes, void *host, size_t host_bytes,
                                uint32_t *tokens, uint64_t *fallbacks, lia_stream_t stream) {
    if (vocab == 0 || !tokens || !logits || !workspace || !host) return LIA_E_ARG;
    if (n == 0) return LIA_OK;
    const size_t records = record_bytes(vocab, n), parts = nucleus_parts(vocab);
    if (workspace_bytes < records || host_bytes < lia_nucleus_host_bytes(vocab, n)) return LIA_E_WORKSPACE;
    const size_t g = (size_t)n * parts;
    const size_t cand_bytes = align_up(g * kSlots * 8, 256), norm_bytes = align_up(g * 16, 256);
    uint8_t *ws = (uint8_t *)workspace, *hb = (uint8_t *)host;
    uint64_t *cand = (uint64_t *)ws;
    double *norm = (double *)(ws + cand_bytes);
    double *temps = (double *)(ws + cand_bytes + norm_bytes);
    double *htemps = (double *)(hb + cand_bytes + norm_bytes);
    float *hrow = (float *)(hb + records);
    RowSummary *sums = (RowSummary *)(ws + records);
    const bool summed = summarised(vocab) && workspace_bytes >= lia_nucleus_workspace_bytes(vocab, n);
    for (uint32_t i = 0; i < n; i++)
        if (samplers && samplers[i] && positions) lia_sampler_set_position(samplers[i], positions[i]);
    temperatures_for(n, samplers, htemps);
    hipStream_t s = (hipStream_t)stream;
    if (hipMemcpyAsync(temps, htemps, (size_t)n * 8, hipMemcpyHostToDevice, s) != hipSuccess)
        return LIA_E_HIP;
    int st = lia_nucleus_candidates(vocab, n, temps, logits, cand, norm, stream);
    if (st) {
        (void)hipStreamSynchronize(s);
        return st;
    }
    // the rows' summaries down (they fit where the records would go), or every part record
    if (summed) {
        const hipError_t e =
            parts * kSlots <= 8 * kRowThreads
                ? launch<nucleus_rows_kernel<8>>(dim3(n), dim3(kRowThreads), 0, s, (uint32_t)parts, temps, cand, norm, sums)
                : launch<nucleus_rows_kernel<16>>(dim3(n), dim3(kRowThreads), 0, s, (uint32_t)parts, temps, cand, norm, sums);
        if (e != hipSuccess) {
            (void)hipStreamSynchronize(s);
            return LIA_E_HIP;
        }
    }
    if (hipMemcpyAsync(hb, summed ? (const void *)sums : ws, summed ? n * sizeof(RowSummary) : cand_bytes + norm_bytes,
                       hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
        return LIA_E_HIP;
    auto down = [&](void *dst, const void *src, size_t bytes) {
        return hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s) == hipSuccess &&
               hipStreamSynchronize(s) == hipSuccess;
    };
    std::vector<Cand> c;
    std::vector<Entry> d;
    std::vector<float> row;
    for (uint32_t r = 0; r < n; r++) {
        auto fetch = [&](float *dst) {
            if (!down(hrow, logits + (size_t)r * vocab, (size_t)vocab * 4)) return (int)LIA_E_HIP;
            memcpy(dst, hrow, (size_t)vocab * 4);
            return (int)LIA_OK;
        };
        lia_sampler *sp = samplers ? samplers[r] : nullptr;
        int st = 2;
        if (summed) st = sample_summary(vocab, sp, ((const RowSummary *)hb)[r], c, d, row, tokens + r, fallbacks, fetch);
        if (st == 2) {
            const uint64_t *rc = (const uint64_t *)hb + r * parts * kSlots;
            const double *rn = (const double *)(hb + cand_bytes) + r * parts * 2;
            if (summed) { // this row's records, through the full-row buffer (4 KB a part)
                uint64_t *hc = (uint64_t *)hrow;
                double *hn = (double *)(hc + parts * kSlots);
                if (!down(hc, cand + r * parts * kSlots, parts * kSlots * 8) || !down(hn, norm + r * parts * 2, parts * 16))
                    return LIA_E_HIP;
                rc = hc;
                rn = hn;
            }
            st = sample_parts(vocab, sp, htemps[r], rc, rn, c, d, row, tokens + r, fallbacks, fetch);
        }
        if (st) return st;
    }
    return LIA_OK;
}
