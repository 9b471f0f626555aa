// Index build on the GPU (build_index.cu:258-363, quantization.cpp:32-193,
// ivf_pg.cpp:110-126): rotation and one-bit / full-code encoding of every
// token and the cluster-ordered layout.
// The arithmetic mirrors the host encoder operation for operation (the same
// fused multiply-adds, the same sequential sums, the same event order in
// best_rescale_factor) so both builds produce identical bytes.
#include "common.hpp"
#include "kernels.hpp"
#include "rotate.hpp"

#include <hipcub/hipcub.hpp>

namespace chimera {

namespace {

struct TightStart {
    float of[9];  // by ex_bits
};
constexpr TightStart kTightStartValues = {{0.F, 0.15F, 0.20F, 0.52F, 0.59F, 0.71F, 0.75F, 0.77F, 0.81F}};
__constant__ TightStart kTightStart = kTightStartValues;

// The rescale search's range of t in units of 1 / max |o|, the least spacing
// of one dimension's events.
constexpr double rescale_spacings(int ex_bits) {
    return ((1 << ex_bits) + 9) * (1.0 - static_cast<double>(kTightStartValues.of[ex_bits]));
}
constexpr double most_rescale_spacings() {
    double most = 0.0;
    for (int e = 1; e <= 7; ++e) most = rescale_spacings(e) > most ? rescale_spacings(e) : most;
    return most;
}

__device__ __forceinline__ uint64_t shfl_xor_u64(uint64_t v, int m) {
    const uint32_t lo = __shfl_xor(static_cast<uint32_t>(v), m, kWave);
    const uint32_t hi = __shfl_xor(static_cast<uint32_t>(v >> 32), m, kWave);
    return (static_cast<uint64_t>(hi) << 32) | lo;
}

__device__ __forceinline__ uint64_t wave_min_u64(uint64_t v) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) {
        const uint64_t o = shfl_xor_u64(v, m);
        v = o < v ? o : v;
    }
    return v;
}

__device__ __forceinline__ int wave_sum_i32(int v) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, kWave);
    return v;
}

// Wave reductions on lane exchanges of the vector ALU: DPP within a row of
// 16 lanes (after the first two steps the quads are uniform, so the mirrors
// act as exchanges), then the lane-swap instructions.
template <int kCtrl>
__device__ __forceinline__ float dpp_f32(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), kCtrl, 0xF, 0xF, true));
}
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppHalfMirror = 0x141, kDppMirror = 0x140;

__device__ __forceinline__ float wave_all_max(float v) {
    v = fmaxf(v, dpp_f32<kDppXor1>(v));
    v = fmaxf(v, dpp_f32<kDppXor2>(v));
    v = fmaxf(v, dpp_f32<kDppHalfMirror>(v));
    v = fmaxf(v, dpp_f32<kDppMirror>(v));
    return wave_max_xor32(wave_max_xor16(v));
}

// v and the value of lane l ^ 16 (or l ^ 32), in some order
__device__ __forceinline__ float2 swap16(float v) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return make_float2(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float2 swap32(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return make_float2(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

__device__ __forceinline__ float wave_all_sum(float v) {
    v += dpp_f32<kDppXor1>(v);
    v += dpp_f32<kDppXor2>(v);
    v += dpp_f32<kDppHalfMirror>(v);
    v += dpp_f32<kDppMirror>(v);
    const float2 a = swap16(v);
    const float2 b = swap32(a.x + a.y);
    return b.x + b.y;
}

__device__ __forceinline__ double join_f64(int lo, int hi) { return __hiloint2double(hi, lo); }

template <int kCtrl>
__device__ __forceinline__ double dpp_f64(double v) {  // 0 from lanes outside the row
    return join_f64(__builtin_amdgcn_update_dpp(0, __double2loint(v), kCtrl, 0xF, 0xF, false),
                    __builtin_amdgcn_update_dpp(0, __double2hiint(v), kCtrl, 0xF, 0xF, false));
}

__device__ __forceinline__ double readlane_f64(double v, int lane) {
    return join_f64(__builtin_amdgcn_readlane(__double2loint(v), lane),
                    __builtin_amdgcn_readlane(__double2hiint(v), lane));
}

// inclusive prefix sums over the wave's lanes (as wave_inclusive_scan)
__device__ __forceinline__ double wave_scan_f64(double v, int l) {
    v += dpp_f64<0x111>(v);
    v += dpp_f64<0x112>(v);
    v += dpp_f64<0x114>(v);
    v += dpp_f64<0x118>(v);
    const double r0 = readlane_f64(v, 15), r1 = readlane_f64(v, 31), r2 = readlane_f64(v, 47);
    const int row = l >> 4;
    double before = row >= 1 ? r0 : 0.0;
    before += row >= 2 ? r1 : 0.0;
    before += row >= 3 ? r2 : 0.0;
    return v + before;
}

__device__ __forceinline__ double wave_all_max_f64(double v) {
    auto up = [](double x, double y) { return x > y ? x : y; };
    v = up(v, dpp_f64<kDppXor1>(v));
    v = up(v, dpp_f64<kDppXor2>(v));
    v = up(v, dpp_f64<kDppHalfMirror>(v));
    v = up(v, dpp_f64<kDppMirror>(v));
    const double a = readlane_f64(v, 0), b = readlane_f64(v, 16), c = readlane_f64(v, 32), d = readlane_f64(v, 48);
    return up(up(a, b), up(c, d));
}

// 32-bit word o of the W-bit packing of 128 raw codes held as 32 words of
// four (packing_rabitqplus_code, pack_excode.hpp; the host pack_codes states
// the same layouts): every layout places runs of four consecutive
// dimensions in four consecutive bytes.
__device__ __forceinline__ uint32_t pack_word(const uint32_t* r, int W, int o) {
    constexpr uint32_t m4 = 0x0F0F0F0Fu, m2 = 0x03030303u;
    switch (W) {
        case 2: {
            const uint32_t* b = r + 4 * o;
            return (b[0] & m2) | (b[1] & m2) << 2 | (b[2] & m2) << 4 | (b[3] & m2) << 6;
        }
        case 4: {
            const uint32_t* b = r + 4 * (o >> 1) + (o & 1);
            return (b[0] & m4) | (b[2] & m4) << 4;
        }
        case 6: {
            const uint32_t* b = r + 4 * (o / 3);
            const int m = o % 3;
            if (m < 2) return (b[m] & m4) | (b[2 + m] & m4) << 4;
            return ((b[0] >> 4) & m2) | ((b[1] >> 4) & m2) << 2 | ((b[2] >> 4) & m2) << 4 | ((b[3] >> 4) & m2) << 6;
        }
        case 8:
            return r[o];
        default: {  // 3, 5, 7: 64-dimension blocks, top bits in the last two words
            const int bb = 2 * W;
            const uint32_t* b = r + 16 * (o / bb);
            const int m = o % bb;
            if (m >= bb - 2) {
                const int k = m - (bb - 2);
                uint32_t v = 0;
#pragma unroll
                for (int g = 0; g < 8; ++g) v |= ((b[2 * g + k] >> (W - 1)) & 0x01010101u) << g;
                return v;
            }
            if (W == 3) return (b[m] & m2) | (b[4 + m] & m2) << 2 | (b[8 + m] & m2) << 4 | (b[12 + m] & m2) << 6;
            if (W == 5) {
                const uint32_t* h = b + 8 * (m >> 2) + (m & 3);
                return (h[0] & m4) | (h[4] & m4) << 4;
            }
            const int part = m >> 2, k = m & 3;  // W == 7
            return (b[4 * part + k] & 0x3F3F3F3Fu) | ((b[12 + k] >> (2 * part)) & m2) << 6;
        }
    }
}

// ---- the rescale factor of the full code (best_rescale_factor,
// quantization.cpp:62-119) ----
//
// A token's codes grow one dimension at a time along the events t = u / a_i
// (dimension i reaches code u), in (t, i) order; after each event the
// similarity is num / sqrt(den), num the sum of (code + 1/2) a_i and den the
// sum of (code + 1/2)^2, and the factor is the t of the first event with the
// largest one. Lane l of the token's wave owns dimensions 2l and 2l + 1, so
// that equal times resolve to the lower dimension.

// What a lane needs of its two dimensions: |o_i|, and the code before the
// first event.
struct RescaleLane {
    float oa, ob;
    int ca, cb;
};

// Event by event: each step takes the wave's earliest event.
__device__ double rescale_sequential(const RescaleLane& in, const float* sabs, double t_start, double t_end, double den,
                                     int top, uint32_t* status, int l) {
    double num = 0.0;
    if (l == 0) {
        for (int i = 0; i < kDim; ++i) {
            const double o = static_cast<double>(sabs[i]);
            const int c = static_cast<int>(fma(t_start, o, 1e-5));
            num = fma(static_cast<double>(c) + 0.5, o, num);
        }
    }
    num = __shfl(num, 0, kWave);
    int ca = in.ca, cb = in.cb;
    double ta = static_cast<double>(ca + 1) / static_cast<double>(in.oa);
    double tb = static_cast<double>(cb + 1) / static_cast<double>(in.ob);
    bool pa = true, pb = true;
    double max_ip = 0.0, tbest = 0.0;
    const int max_events = kDim * (top + 2) + 1;
    int it = 0;
    for (; it < max_events; ++it) {
        const uint64_t ka = pa ? static_cast<uint64_t>(__double_as_longlong(ta)) : ~0ull;
        const uint64_t kb = pb ? static_cast<uint64_t>(__double_as_longlong(tb)) : ~0ull;
        const bool sel_b = kb < ka;
        const uint64_t key = sel_b ? kb : ka;
        const uint64_t kmin = wave_min_u64(key);
        if (kmin == ~0ull) break;
        const int win = __builtin_ctzll(__ballot(key == kmin));
        const int u = __shfl((sel_b ? cb : ca) + 1, win, kWave);
        const float o = __shfl(sel_b ? in.ob : in.oa, win, kWave);
        const double cur_t = __longlong_as_double(static_cast<long long>(kmin));
        den += static_cast<double>(2 * u);
        num += static_cast<double>(o);
        const double cur_ip = num / sqrt(den);
        if (cur_ip > max_ip) {
            max_ip = cur_ip;
            tbest = cur_t;
        }
        if (l == win) {
            bool keep = false;
            double tn = 0.0;
            if (u < top) {
                tn = static_cast<double>(u + 1) / static_cast<double>(o);
                keep = tn < t_end;
            }
            if (sel_b) {
                cb = u;
                pb = keep;
                if (keep) tb = tn;
            } else {
                ca = u;
                pa = keep;
                if (keep) ta = tn;
            }
        }
    }
    if (it == max_events && l == 0) atomicOr(status, 2u);
    return tbest;
}

// All events at once. They fall into kBins (256 or 512) intervals of [t_start, t_end)
// and one for t >= t_end (each dimension's first event is taken wherever it
// lies); the sums per interval, and a wave scan over them, give the state
// (num, den) at the end of every interval. Inside an interval that starts at
// time tl with state (n, d) an event that adds x to num adds 2 t x >= 2 tl x
// to den, so its states lie at or below the curve (n + x)^2 / (d + 2 tl x),
// 0 <= x <= X (X the interval's sum). That curve falls and then rises (the
// sign of its slope is that of d - tl n + tl x), so max(n^2 / d,
// (n + X)^2 / (d + 2 tl X)) bounds the interval, and only the intervals
// whose bound reaches the best interval end are stepped through: 1.3 to 2.8
// of the 257 on Gaussian tokens (2.2 of 513 at ex_bits 7).
//
// The sums are the sequential ones: the caller has checked that every
// partial sum of num is a multiple of a power of two below 2^53 of them, so
// no addition rounds in any order (den is a sum of integers). The comparison
// of squares uses a reciprocal good to 1e-14 and keeps all within 1e-12 of
// the best, which then compare by num / sqrt(den) as the sequential search.
//
// The time u / a is the correctly rounded quotient: with y = RN(1 / a),
// q = RN(u y) and the exact remainder r = u - a q, q + r y differs from
// u / a by less than 2^-103 of it (Markstein's correction), and a quotient of
// an 8-bit by a 24-bit number is never that close to a rounding boundary of
// 53 bits.
//
// An interval is narrower than 1 / max a = the least spacing of one
// dimension's events (the range is at most 31.5 spacings, at ex_bits 7), so a
// dimension has at most one event in it.
//
// The walk takes as many steps as the lane with the most events, so its lanes
// do not take the dimensions that they own: the dimensions are sorted by event
// count (a counting sort in the intervals' memory) and lane l takes the l-th
// from either end. On Gaussian tokens at ex_bits 7 that is 28 steps instead
// of 42 (11 to 7.5 at ex_bits 4): 2.9M tokens 25.2 -> 23.8 ms, 0.88M at
// ex_bits 4 3.56 -> 3.51 ms.
constexpr int kOrderKeys = 32;  // counts past 31 (of at most 33) share a key: the order only evens out the walk
template <int kBins>
union RescaleBins {
    struct {
        double sum[kBins + 1];    // sum of a_i over the interval's events
        uint32_t cu[kBins + 1];   // events << 16 | sum of u
    };
    struct {  // before the walk: the dimensions by event count
        double y[kDim];
        float a[kDim];
        int code[kDim], events[kDim];
        int head[kOrderKeys];
    } order;
};

template <int kBins>
__device__ double rescale_binned(const RescaleLane& in, RescaleBins<kBins>& bins, double t_start, double t_end, double num0,
                                 double den0, int top, int l) {
    static_assert(2.0 * most_rescale_spacings() < kBins, "at most one event of a dimension in an interval");
    constexpr int kPerLane = kBins / kWave;
    const double ya = in.oa > 0.0f ? 1.0 / static_cast<double>(in.oa) : 0.0;
    const double yb = in.ob > 0.0f ? 1.0 / static_cast<double>(in.ob) : 0.0;
    const double width = (t_end - t_start) * (1.0 / kBins);
    const double scale = 1.0 / width;
    auto time_of = [](int u, float a, double y) {
        const double du = static_cast<double>(u), da = static_cast<double>(a);
        const double q = du * y;
        const double r = fma(-da, q, du);
        return a > 0.0f ? fma(r, y, q) : INFINITY;
    };
    // the interval of a time: non-decreasing in t
    auto bin_of = [&](double t) {
        if (!(t < t_end)) return kBins;
        const int b = static_cast<int>((t - t_start) * scale);
        return b < 0 ? 0 : (b < kBins ? b : kBins - 1);
    };
    // A dimension's events are u = c + 1 .. last: the first wherever it lies,
    // the others while u <= top and u / a < t_end. The largest u below t_end
    // is within one of t_end a, so the counts are known before the walk, which
    // then has one branch a step.
    auto events_of = [&](float a, double y, int c) {
        int last = static_cast<int>(t_end * static_cast<double>(a));
        if (!(time_of(last, a, y) < t_end))
            --last;
        else if (time_of(last + 1, a, y) < t_end)
            ++last;
        last = last < top ? last : top;
        return (last > c + 1 ? last : c + 1) - c;
    };
    {
        const int own_a = events_of(in.oa, ya, in.ca), own_b = events_of(in.ob, yb, in.cb);
        const int key_a = min(max(own_a, 0), kOrderKeys - 1), key_b = min(max(own_b, 0), kOrderKeys - 1);
        if (l < kOrderKeys) bins.order.head[l] = 0;
        wave_lds_sync();
        int at_a = atomicAdd(&bins.order.head[key_a], 1);
        int at_b = atomicAdd(&bins.order.head[key_b], 1);
        wave_lds_sync();
        const int keys = l < kOrderKeys ? bins.order.head[l] : 0;
        const int before = wave_inclusive_scan(keys) - keys;
        if (l < kOrderKeys) bins.order.head[l] = before;
        wave_lds_sync();
        at_a += bins.order.head[key_a];
        at_b += bins.order.head[key_b];
        auto place = [&](int at, double y, float a, int c, int n) {
            bins.order.y[at] = y;
            bins.order.a[at] = a;
            bins.order.code[at] = c;
            bins.order.events[at] = n;
        };
        place(at_a, ya, in.oa, in.ca, own_a);
        place(at_b, yb, in.ob, in.cb, own_b);
        wave_lds_sync();
        const int lo = l, hi = kDim - 1 - l;
        const double y0 = bins.order.y[lo], y1 = bins.order.y[hi];
        const float a0 = bins.order.a[lo], a1 = bins.order.a[hi];
        const int c0 = bins.order.code[lo], c1 = bins.order.code[hi];
        const int n0 = bins.order.events[lo];
        const int total = n0 + bins.order.events[hi];
        wave_lds_sync();
        for (int b = l; b < kBins + 1; b += kWave) {
            bins.sum[b] = 0.0;
            bins.cu[b] = 0u;
        }
        wave_lds_sync();
        const int trips = static_cast<int>(wave_all_max(static_cast<float>(total)));
        for (int i = 0; i < trips; ++i) {
            const bool second = i >= n0;  // one dimension's events, then the other's
            const float a = second ? a1 : a0;
            const int u = i + (second ? c1 + 1 - n0 : c0 + 1);
            const int b = bin_of(time_of(u, a, second ? y1 : y0));
            if (i < total) {
                atomicAdd(&bins.sum[b], static_cast<double>(a));
                atomicAdd(&bins.cu[b], (1u << 16) + static_cast<uint32_t>(u));
            }
        }
    }
    wave_lds_sync();
    // interval ends: lane l owns kPerLane consecutive intervals
    double sums[kPerLane];
    uint32_t cu[kPerLane];
    double own = 0.0;
    int own_u = 0;
#pragma unroll
    for (int k = 0; k < kPerLane; ++k) {
        sums[k] = bins.sum[kPerLane * l + k];
        cu[k] = bins.cu[kPerLane * l + k];
        own += sums[k];
        own_u += static_cast<int>(cu[k] & 0xFFFFu);
    }
    const double incl = wave_scan_f64(own, l);
    const int incl_u = wave_inclusive_scan(own_u);
    const double late_n = num0 + readlane_f64(incl, kWave - 1);
    const int late_du = __builtin_amdgcn_readlane(incl_u, kWave - 1);
    const double late_d = den0 + static_cast<double>(2 * late_du);
    auto square_ratio = [](double n, double d) {  // n^2 / d, relative error below 1e-14
        double y = __builtin_amdgcn_rcp(d);
        y = fma(fma(-d, y, 1.0), y, y);
        y = fma(fma(-d, y, 1.0), y, y);
        return n * n * y;
    };
    const double n_first = num0 + (incl - own);
    const int u_first = incl_u - own_u;
    double best = 0.0;
    double bound[kPerLane];  // of the interval's states (its end state for one event, 0 for none)
    {
        double n = n_first;
        int du = u_first;
        double g = square_ratio(n, den0 + static_cast<double>(2 * du));
#pragma unroll
        for (int k = 0; k < kPerLane; ++k) {
            const uint32_t count = cu[k] >> 16;
            const double d = den0 + static_cast<double>(2 * du);
            const double n_end = n + sums[k];
            du += static_cast<int>(cu[k] & 0xFFFFu);
            const double g_end = square_ratio(n_end, den0 + static_cast<double>(2 * du));
            const double tl = t_start + (kPerLane * l + k) * width;
            const double curve = square_ratio(n_end, d + 2.0 * (tl * (1.0 - 1e-12)) * sums[k]);
            const double inside = g > curve ? g : curve;
            bound[k] = count == 0u ? 0.0 : (count == 1u ? g_end : (inside > g_end ? inside : g_end));
            if (count != 0u && g_end > best) best = g_end;
            n = n_end;
            g = g_end;
        }
    }
    const double late_sum = bins.sum[kBins];
    const uint32_t late_cu = bins.cu[kBins];
    const uint32_t late_count = late_cu >> 16;
    double late_bound = 0.0;
    if (late_count != 0u) {
        const double g_end = square_ratio(late_n + late_sum, late_d + static_cast<double>(2 * (late_cu & 0xFFFFu)));
        const double g = square_ratio(late_n, late_d);
        const double curve = square_ratio(late_n + late_sum, late_d + 2.0 * (t_end * (1.0 - 1e-12)) * late_sum);
        const double inside = g > curve ? g : curve;
        late_bound = inside > g_end ? inside : g_end;
        if (g_end > best) best = g_end;
    }
    const double need = wave_all_max_f64(best) * (1.0 - 1e-12);
    uint32_t cand = 0u;
#pragma unroll
    for (int k = 0; k < kPerLane; ++k) cand |= (bound[k] > 0.0 && bound[k] >= need ? 1u : 0u) << k;

    double max_ip = 0.0, tbest = 0.0;
    bool late = late_bound > 0.0 && late_bound >= need;
    for (uint64_t lanes = __ballot(cand != 0u); lanes != 0ull || late;) {
        // the next interval, and the state before it
        int b = kBins, du = late_du;
        double n = late_n;
        if (lanes != 0ull) {
            const int lane = __builtin_ctzll(lanes);
            const uint32_t which = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(cand), lane));
            b = kPerLane * lane + __builtin_ctz(which);
            n = readlane_f64(n_first, lane);
            du = __builtin_amdgcn_readlane(u_first, lane);
            for (int i = kPerLane * lane; i < b; ++i) {
                n += bins.sum[i];
                du += static_cast<int>(bins.cu[i] & 0xFFFFu);
            }
            if (l == lane) cand &= cand - 1u;
            if ((which & (which - 1u)) == 0u) lanes &= lanes - 1ull;
        } else {
            late = false;
        }
        double d = den0 + static_cast<double>(2 * du);
        // a lane's events in it: at most one per dimension
        const double tl = t_start + b * width;
        auto event = [&](float a, double y, int c, int& u) {
            u = c + 1;
            if (b < kBins) {
                const int at = static_cast<int>(tl * static_cast<double>(a));
                u = at > u ? at : u;
            }
            double t = time_of(u, a, y);
            if (b < kBins && bin_of(t) < b && u + 1 <= top) t = time_of(++u, a, y);
            return bin_of(t) == b && (u == c + 1 || u <= top) ? static_cast<uint64_t>(__double_as_longlong(t)) : ~0ull;
        };
        int ua, ub;
        uint64_t ka = event(in.oa, ya, in.ca, ua);
        uint64_t kb = event(in.ob, yb, in.cb, ub);
        for (int it = 0; it < kDim; ++it) {
            const bool sel_b = kb < ka;
            const uint64_t key = sel_b ? kb : ka;
            const uint64_t have = __ballot(key != ~0ull);
            if (have == 0ull) break;
            // one lane left: its time is the earliest
            const int only = __builtin_ctzll(have);
            const uint64_t kmin =
                (have & (have - 1ull)) == 0ull
                    ? static_cast<uint64_t>(__double_as_longlong(readlane_f64(__longlong_as_double(static_cast<long long>(key)), only)))
                    : wave_min_u64(key);
            const int win = __builtin_ctzll(__ballot(key == kmin));
            n += static_cast<double>(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(sel_b ? in.ob : in.oa), win)));
            d += static_cast<double>(2 * __builtin_amdgcn_readlane(sel_b ? ub : ua, win));
            const double cur_ip = n / sqrt(d);
            if (cur_ip > max_ip) {
                max_ip = cur_ip;
                tbest = __longlong_as_double(static_cast<long long>(kmin));
            }
            if (l == win) {
                if (sel_b) kb = ~0ull; else ka = ~0ull;
            }
        }
    }
    return tbest;
}

}  // namespace

// Encodes 32 tokens per block and step: each wave rotates and quantises
// eight of them, a lane per dimension pair, while the sums that the host
// encoder takes in dimension order run a lane per token (three serial chains
// of 128 adds for all 32 tokens at once). Rotated rows and raw codes stay in
// LDS between the phases; rows of 129 floats and 33 code words put a lane
// per token on distinct banks. The packed codes of the 32 tokens are one
// contiguous run of words.
//
// What bounds it is vector-ALU issue of the rescale search (about 2,500
// instructions a token at ex_bits 4, against 0.6 KB of HBM traffic). Measured
// on MI355X: 0.88M tokens at ex_bits 4 in 3.5 ms and 2.9M tokens at ex_bits 7
// in 23.8 ms; one wave per token that took the events one at a time and ran
// the three serial sums on one lane took 63.2 and 659 ms. Four waves per SIMD
// (128 VGPRs) need the 35 KB of LDS that 32 tokens take.
constexpr int kEncTokens = 32;
constexpr int kEncWaves = 4;
template <int kBins>
__global__ __launch_bounds__(kEncWaves * kWave, kBins <= 256 ? 4 : 3) void encode_tokens_kernel(
    const float* __restrict__ emb, int64_t n, int dim, const uint8_t* __restrict__ flips, float fac, int ex_bits,
    uint8_t* __restrict__ codes1, float* __restrict__ f1, uint8_t* __restrict__ full, float* __restrict__ fF,
    uint32_t* __restrict__ status) {
    constexpr int kRow = kDim + 1, kRawRow = kDim / 4 + 1;
    __shared__ float srow[kEncTokens][kRow];
    __shared__ uint32_t sraw[kEncTokens][kRawRow];
    __shared__ float sabs[kEncWaves][kDim];  // the sequential search's copy
    __shared__ float sip[kEncTokens], ssq[kEncTokens];
    __shared__ uint32_t sbad[kEncTokens];
    __shared__ RescaleBins<kBins> bins[kEncWaves];
    __shared__ uint8_t fl[4 * kDim / 8];
    const int l = lane_id();
    const int w = wave_id();
    if (threadIdx.x < 4 * kDim / 8) fl[threadIdx.x] = flips[threadIdx.x];
    __syncthreads();
    const int top = (1 << ex_bits) - 1;
    const int W = ex_bits + 1;
    const bool pow2 = dim >= kDim;
    const int64_t stride = static_cast<int64_t>(gridDim.x) * kEncTokens;
    for (int64_t base = static_cast<int64_t>(blockIdx.x) * kEncTokens; base < n; base += stride) {
        const int nt = static_cast<int>(n - base < kEncTokens ? n - base : kEncTokens);
        for (int i = w; i < nt; i += kEncWaves) {
            const int64_t t = base + i;
            const float* src = emb + t * dim;
            float x0 = l < dim ? src[l] : 0.0f;
            float x1 = l + 64 < dim ? src[l + 64] : 0.0f;
            fht_kac_rotate(x0, x1, fl, fac, pow2, l);
            srow[i][l] = x0;
            srow[i][l + 64] = x1;
            // one-bit code: bit j of the little-endian 128-bit word is o'_j > 0
            const uint64_t m0 = __ballot(x0 > 0.0f);
            const uint64_t m1 = __ballot(x1 > 0.0f);
            if (l == 0) {
                uint4 v;
                v.x = static_cast<uint32_t>(m0);
                v.y = static_cast<uint32_t>(m0 >> 32);
                v.z = static_cast<uint32_t>(m1);
                v.w = static_cast<uint32_t>(m1 >> 32);
                reinterpret_cast<uint4*>(codes1)[t] = v;
            }
        }
        __syncthreads();
        // wave 0: <x_u - 1/2, o'> ; wave 1: |o'|^2 ; both in dimension order
        if (w < 2 && l < nt) {
            float acc = 0.0f;
#pragma unroll 8
            for (int j = 0; j < kDim; ++j) {
                const float r = srow[l][j];
                const float x = (w == 0) ? ((r > 0.0f ? 1.0f : 0.0f) - 0.5F) : r;
                acc = __fmaf_rn(x, r, acc);
            }
            (w == 0 ? sip : ssq)[l] = acc;
        }
        __syncthreads();
        for (int i = w; i < nt; i += kEncWaves) {
            const float xa = srow[i][2 * l], xb = srow[i][2 * l + 1];
            const float norm = sqrtf(ssq[i]);
            RescaleLane in;
            in.oa = norm > 0.0f ? fabsf(xa / norm) : fabsf(xa);
            in.ob = norm > 0.0f ? fabsf(xb / norm) : fabsf(xb);
            const float max_o = wave_all_max(fmaxf(in.oa, in.ob));
            const bool finite = __ballot(!(isfinite(xa) && isfinite(xb))) == 0ull;
            uint16_t* raw = reinterpret_cast<uint16_t*>(sraw[i]) + l;
            if (!finite || !(max_o > 0.0f) || !isfinite(max_o)) {
                // zero or non-finite token: the rescale search is undefined
                if (l == 0) {
                    atomicOr(status, 1u);
                    sbad[i] = 1u;
                }
                *raw = 0;
                continue;
            }
            if (l == 0) sbad[i] = 0u;
            const double t_end = static_cast<double>(top + 10) / static_cast<double>(max_o);
            const double t_start = t_end * static_cast<double>(kTightStart.of[ex_bits]);
            in.ca = static_cast<int>(fma(t_start, static_cast<double>(in.oa), 1e-5));
            in.cb = static_cast<int>(fma(t_start, static_cast<double>(in.ob), 1e-5));
            const double den = static_cast<double>(kDim) * 0.25 +
                               static_cast<double>(wave_sum_i32(in.ca * in.ca + in.ca + in.cb * in.cb + in.cb));
            // num stays below t_end sum a^2 + 1.51 sum a <= 2^e; with every
            // a_i a multiple of 2^(e - 52), every (code + 1/2) a_i and every
            // partial sum is a multiple of 2^(e - 53): exact in any order
            const float most = static_cast<float>(t_end) * wave_all_sum(in.oa * in.oa + in.ob * in.ob) +
                               1.52f * wave_all_sum(in.oa + in.ob);
            const int e = ilogbf(most * 1.001f) + 1;
            const double za = ldexp(static_cast<double>(in.oa), 52 - e), zb = ldexp(static_cast<double>(in.ob), 52 - e);
            const bool exact = max_o >= 0.0625f && max_o <= 1.01f &&
                               __ballot(!(za == trunc(za) && zb == trunc(zb))) == 0ull;
            double tbest;
            if (exact) {
                const double part = (static_cast<double>(in.ca) + 0.5) * static_cast<double>(in.oa) +
                                    (static_cast<double>(in.cb) + 0.5) * static_cast<double>(in.ob);
                const double num = readlane_f64(wave_scan_f64(part, l), kWave - 1);
                tbest = rescale_binned(in, bins[w], t_start, t_end, num, den, top, l);
            } else {
                sabs[w][2 * l] = in.oa;
                sabs[w][2 * l + 1] = in.ob;
                wave_lds_sync();
                tbest = rescale_sequential(in, sabs[w], t_start, t_end, den, top, status, l);
            }
            // quantize_ex + total code (quantization.cpp:121-193)
            int e0 = static_cast<int>(fma(tbest, static_cast<double>(in.oa), 1e-5));
            int e1 = static_cast<int>(fma(tbest, static_cast<double>(in.ob), 1e-5));
            e0 = e0 > top ? top : e0;
            e1 = e1 > top ? top : e1;
            if (xa < 0.0f) e0 = (~e0) & top;
            if (xb < 0.0f) e1 = (~e1) & top;
            e0 += (xa >= 0.0f ? 1 : 0) << ex_bits;
            e1 += (xb >= 0.0f ? 1 : 0) << ex_bits;
            *raw = static_cast<uint16_t>(e0 | (e1 << 8));
        }
        __syncthreads();
        if (w == 0 && l < nt) {
            const float cbf = -(static_cast<float>(1 << ex_bits) - 0.5F);
            float ip = 0.0f;
#pragma unroll 2
            for (int j4 = 0; j4 < kDim / 4; ++j4) {
                const uint32_t c = sraw[l][j4];
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    ip = __fmaf_rn(static_cast<float>((c >> (8 * u)) & 255u) + cbf, srow[l][4 * j4 + u], ip);
            }
            f1[base + l] = 1.0F / sip[l];
            fF[base + l] = sbad[l] ? 0.0f : 1.0F / ip;
        }
        const int words = 4 * W;
        uint32_t* out = reinterpret_cast<uint32_t*>(full + base * (16 * W));
        for (int o = static_cast<int>(threadIdx.x); o < nt * words; o += kEncWaves * kWave)
            out[o] = pack_word(sraw[o / words], W, o % words);
        __syncthreads();
    }
}

// Rows src[ids[r]] (dim floats) zero-padded to 128, optionally rotated.
__global__ __launch_bounds__(256) void gather_rows_kernel(const float* __restrict__ src, int dim,
                                                          const int64_t* __restrict__ ids, int64_t nrows,
                                                          const uint8_t* __restrict__ flips, float fac, int rotate,
                                                          float* __restrict__ out) {
    __shared__ uint8_t fl[4 * kDim / 8];
    const int l = lane_id();
    if (threadIdx.x < 4 * kDim / 8) fl[threadIdx.x] = rotate ? flips[threadIdx.x] : 0;
    __syncthreads();
    const int64_t r = static_cast<int64_t>(blockIdx.x) * 4 + wave_id();
    if (r >= nrows) return;
    const float* s = src + (ids ? ids[r] : r) * dim;
    float x0 = l < dim ? s[l] : 0.0f;
    float x1 = l + 64 < dim ? s[l + 64] : 0.0f;
    if (rotate) fht_kac_rotate(x0, x1, fl, fac, dim >= kDim, l);
    out[r * kDim + l] = x0;
    out[r * kDim + l + 64] = x1;
}

__global__ void iota_u32_kernel(uint32_t* __restrict__ v, int64_t n) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) v[i] = static_cast<uint32_t>(i);
}

__global__ void invert_kernel(const uint32_t* __restrict__ inv, int64_t n, uint32_t* __restrict__ pos) {
    const int64_t p = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (p < n) pos[inv[p]] = static_cast<uint32_t>(p);
}

// cluster_pos[c] = first position of cluster c in the sorted assignments.
__global__ void cluster_bounds_kernel(const uint32_t* __restrict__ sorted, int64_t n, int64_t k,
                                      uint64_t* __restrict__ cluster_pos) {
    const int64_t c = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (c > k) return;
    int64_t lo = 0, hi = n;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (static_cast<int64_t>(sorted[mid]) < c) lo = mid + 1; else hi = mid;
    }
    cluster_pos[c] = static_cast<uint64_t>(lo);
}

__global__ void token_doc_kernel(const int32_t* __restrict__ doc_ptrs, int64_t m, int32_t* __restrict__ token_doc) {
    const int64_t d = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (d >= m) return;
    for (int32_t t = doc_ptrs[d]; t < doc_ptrs[d + 1]; ++t) token_doc[t] = static_cast<int32_t>(d);
}

// reorder_by_cluster (build_index.cu:328-363)
__global__ void reorder_kernel(const uint32_t* __restrict__ inv, int64_t n, const uint8_t* __restrict__ codes_tok,
                               const float* __restrict__ f1_tok, const int32_t* __restrict__ token_doc,
                               uint8_t* __restrict__ codes_clu, float* __restrict__ f1_clu,
                               int32_t* __restrict__ doc_clu) {
    const int64_t p = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const uint32_t t = inv[p];
    reinterpret_cast<uint4*>(codes_clu)[p] = reinterpret_cast<const uint4*>(codes_tok)[t];
    f1_clu[p] = f1_tok[t];
    doc_clu[p] = token_doc[t];
}

// ---- launchers ----

namespace {
unsigned blocks_for(int64_t n, int per) { return static_cast<unsigned>((n + per - 1) / per); }
}  // namespace

hipError_t launch_encode_tokens(hipStream_t s, const float* emb, int64_t n, int dim, const uint8_t* flips,
                                int ex_bits, int num_cus, uint8_t* codes1, float* f1, uint8_t* full, float* fF,
                                uint32_t* status) {
    if (n == 0) return hipSuccess;
    const int trunc = dim >= kDim ? kDim : 64;
    const float fac = 1.0F / sqrtf(static_cast<float>(trunc));
    const int64_t want = static_cast<int64_t>(num_cus) * 16;
    const unsigned grid = static_cast<unsigned>(std::min<int64_t>((n + kEncTokens - 1) / kEncTokens, want));
    auto encode = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(kEncWaves * kWave), 0, s, emb, n, dim, flips, fac, ex_bits, codes1, f1,
                           full, fF, status);
    };
    // More intervals leave fewer events to step through and cost a longer
    // scan and a wave less per SIMD, which pays at 8-bit codes only. 2.9M
    // tokens with 256 and with 512, ms, by ex_bits: 4 9.68 and 11.10, 5 10.73
    // and 11.88, 6 15.04 and 15.17, 7 26.92 and 23.06; of 96 dimensions 6
    // 14.29 and 14.43, 7 26.14 and 22.12.
    if (ex_bits >= 7)
        encode(encode_tokens_kernel<512>);
    else
        encode(encode_tokens_kernel<256>);
    return hipGetLastError();
}

hipError_t launch_gather_rows(hipStream_t s, const float* src, int dim, const int64_t* ids, int64_t nrows,
                              const uint8_t* flips, bool rotate, float* out) {
    if (nrows == 0) return hipSuccess;
    const int trunc = dim >= kDim ? kDim : 64;
    const float fac = 1.0F / sqrtf(static_cast<float>(trunc));
    hipLaunchKernelGGL(gather_rows_kernel, dim3(blocks_for(nrows, 4)), dim3(256), 0, s, src, dim, ids, nrows, flips,
                       fac, rotate ? 1 : 0, out);
    return hipGetLastError();
}

hipError_t launch_sort_assignments(hipStream_t s, const uint32_t* labels, int64_t n, int64_t k, uint32_t* keys_out,
                                   uint32_t* vals_in, uint32_t* vals_out, void* temp, size_t* temp_bytes) {
    int end_bit = 1;
    while ((int64_t{1} << end_bit) < k) ++end_bit;
    if (temp == nullptr)
        return hipcub::DeviceRadixSort::SortPairs(nullptr, *temp_bytes, labels, keys_out, vals_in, vals_out,
                                                  static_cast<int>(n), 0, end_bit, s);
    hipLaunchKernelGGL(iota_u32_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, s, vals_in, n);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return hipcub::DeviceRadixSort::SortPairs(temp, *temp_bytes, labels, keys_out, vals_in, vals_out,
                                              static_cast<int>(n), 0, end_bit, s);
}

hipError_t launch_invert(hipStream_t s, const uint32_t* inv, int64_t n, uint32_t* pos) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(invert_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, s, inv, n, pos);
    return hipGetLastError();
}

hipError_t launch_layout(hipStream_t s, const uint32_t* sorted_keys, const uint32_t* inv, int64_t n, int64_t k,
                         const int32_t* doc_ptrs, int64_t m, const uint8_t* codes_tok, const float* f1_tok,
                         int32_t* token_doc, uint64_t* cluster_pos, uint8_t* codes_clu, float* f1_clu,
                         int32_t* doc_clu) {
    hipLaunchKernelGGL(cluster_bounds_kernel, dim3(blocks_for(k + 1, 256)), dim3(256), 0, s, sorted_keys, n, k,
                       cluster_pos);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(token_doc_kernel, dim3(blocks_for(m, 256)), dim3(256), 0, s, doc_ptrs, m, token_doc);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(reorder_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, s, inv, n, codes_tok, f1_tok, token_doc,
                       codes_clu, f1_clu, doc_clu);
    return hipGetLastError();
}

}  // namespace chimera
