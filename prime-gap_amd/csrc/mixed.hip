// mixed.hip -- pgap_prp_batch_mixed: bucket the numbers, queue tiles widest
// first and run the kernels of mixed_impl.h (matrix-core numbers and one-lane
// buckets side by side on two streams).
#include <algorithm>
#include <cmath>
#include <vector>

#include "engine_impl.h"
#include "mixed_impl.h"

using namespace pgap;

static pgap_status mixed_once(pgap_engine *e, const uint32_t *words, const uint64_t *offset, const uint32_t *limbs,
                              size_t count, pgap_test kind, const uint32_t *bases, uint32_t nbases,
                              uint8_t *verdict);

// Several strong-PRP bases: the first base runs on every number, each later
// base only on the numbers that passed so far (a few percent of sieved
// candidates), so the widest lane of a wavefront never carries the others
// through bases they have already failed.
extern "C" pgap_status pgap_prp_batch_mixed(pgap_engine *e, const uint32_t *words, const uint64_t *offset,
                                            const uint32_t *limbs, size_t count, pgap_test kind,
                                            const uint32_t *bases, uint32_t nbases, uint8_t *verdict) {
    if (!e || kind != PGAP_SPRP || nbases <= 1 || !bases || nbases > (uint32_t)kMaxBases || !verdict || !offset ||
        !limbs)
        return mixed_once(e, words, offset, limbs, count, kind, bases, nbases, verdict);
    pgap_status st = mixed_once(e, words, offset, limbs, count, kind, bases, 1, verdict);
    for (uint32_t k = 1; k < nbases && st == PGAP_OK; ++k) {
        std::vector<uint64_t> off;
        std::vector<uint32_t> lim;
        std::vector<size_t> at;
        for (size_t i = 0; i < count; ++i)
            if (verdict[i]) {
                off.push_back(offset[i]);
                lim.push_back(limbs[i]);
                at.push_back(i);
            }
        if (at.empty()) break;
        std::vector<uint8_t> v(at.size());
        st = mixed_once(e, words, off.data(), lim.data(), at.size(), kind, bases + k, 1, v.data());
        for (size_t j = 0; j < at.size() && st == PGAP_OK; ++j) verdict[at[j]] = v[j];
    }
    return st;
}

static pgap_status mixed_once(pgap_engine *e, const uint32_t *words, const uint64_t *offset, const uint32_t *limbs,
                              size_t count, pgap_test kind, const uint32_t *bases, uint32_t nbases,
                              uint8_t *verdict) {
    if (!e) return PGAP_E_ARG;
    if (!e->ready) return PGAP_E_STATE;
    if (count == 0) return PGAP_OK;
    if (!words || !offset || !limbs || !verdict || count > 0xfffffff0u) {
        e->set_error("pgap_prp_batch_mixed: bad arguments");
        return PGAP_E_ARG;
    }
    Bases bs{};
    if (kind == PGAP_SPRP) {
        if (nbases == 0 || nbases > (uint32_t)kMaxBases || !bases) {
            e->set_error("SPRP needs 1..%d bases", kMaxBases);
            return PGAP_E_ARG;
        }
        bs.n = nbases;
        for (uint32_t i = 0; i < nbases; ++i) {
            if (bases[i] < 2 || bases[i] > 63) {
                e->set_error("SPRP base %u outside [2, 63]", bases[i]);
                return PGAP_E_ARG;
            }
            bs.b[i] = bases[i];
        }
        if (nbases > 1) {  // the kernel tests bases.b[0]; pgap_prp_batch_mixed stages the others
            e->set_error("pgap_prp_batch_mixed: one base per persistent launch");
            return PGAP_E_ARG;
        }
    } else if (kind != PGAP_FERMAT2) {
        e->set_error("pgap_prp_batch_mixed runs FERMAT2 or SPRP (kind %d)", (int)kind);
        return PGAP_E_ARG;
    }
    // bucket per number: the smallest digit count whose bound covers it,
    // headroom below R = 2^(28 digits) as the one-lane variants need, or the
    // last for numbers wider than one lane takes
    constexpr int N1 = MixedOneLane::n;
    const int slack1 = kind == PGAP_FERMAT2 ? 4 : 8 + (int)(select_bits(KIND_SPRP, 0, bs));
    const int widest = kMixedMaxBits - (kind == PGAP_FERMAT2 ? 4 : 8);
    struct Bucket {
        std::vector<uint32_t> rows, bits;
        uint32_t most = 0;  // widest row
    };
    std::vector<Bucket> bucket(N1 + 1);
    size_t total_words = 0;
    for (size_t i = 0; i < count; ++i) {
        const uint32_t *w = words + offset[i];
        uint32_t bits = 0;
        for (int j = (int)limbs[i] - 1; j >= 0; --j)
            if (w[j]) {
                bits = 32u * (uint32_t)j + (32u - (uint32_t)__builtin_clz(w[j]));
                break;
            }
        bits = std::max(bits, 2u);
        int b = 0;
        while (b < N1 && 28 * MixedOneLane::digits[b] - slack1 < (int)bits) ++b;
        if ((int)bits > widest) {
            e->set_error("pgap_prp_batch_mixed: number %zu has %u bits, above the widest bucket (%d)", i, bits, widest);
            return PGAP_E_TOO_LARGE;
        }
        bucket[(size_t)b].rows.push_back((uint32_t)i);
        bucket[(size_t)b].bits.push_back(bits);
        bucket[(size_t)b].most = std::max(bucket[(size_t)b].most, bits);
        total_words = std::max<size_t>(total_words, offset[i] + limbs[i]);
    }
    // Buckets below `cut` go to the persistent kernel in tiles of 64, widest
    // first (order[1]); the other rows to the matrix cores by container, widest
    // first (order[0]).  The one-lane tiles together take the widest one's time
    // or the device's for their sum, whichever is more, so a narrower bucket
    // costs nothing beside a wide one; rows on the matrix cores add up.  Chosen
    // bucket by bucket instead (each against a round of its own), five buckets
    // that each just stay below a round took 67.9 ms against 49.3 in tiles.
    const double simds = 4.0 * e->num_cus;
    int cut = 0;
    double least = 0;
    for (int c = N1; c >= 0; --c) {
        if (c == 0 && !bucket[0].rows.empty() && bucket[0].most < kMatrixMinBits) break;
        double longest = 0, tiles = 0, matrix = 0;
        for (int b = 0; b < N1; ++b) {
            const Bucket &k = bucket[(size_t)b];
            if (k.rows.empty()) continue;
            const double tile = kTileCycles[b] * k.most, rows = (double)k.rows.size();
            if (b < c) {
                longest = std::max(longest, tile);
                tiles += std::ceil(rows / 64) * tile;
            } else {
                matrix += rows * kMixedMatrixCycles[find_matrix(KIND_FERMAT2, (int)k.most)->blocks] * k.most;
            }
        }
        const double time = std::max(longest, tiles / simds) + matrix / simds;
        if (c == N1 || time < least) {
            least = time;
            cut = c;
        }
    }
    std::vector<uint32_t> order[2], container[kMixedContainers];
    std::vector<uint8_t> tile_bucket;
    for (int b = N1; b >= 0; --b) {
        const Bucket &k = bucket[(size_t)b];
        if (b >= cut) {
            for (size_t i = 0; i < k.rows.size(); ++i)
                container[find_matrix(KIND_FERMAT2, (int)k.bits[i])->blocks - 1].push_back(k.rows[i]);
            continue;
        }
        for (size_t i = 0; i < k.rows.size(); i += 64) {
            tile_bucket.push_back((uint8_t)b);
            for (size_t l = 0; l < 64; ++l)
                order[1].push_back(i + l < k.rows.size() ? k.rows[i + l] : 0xffffffffu);
        }
    }
    MixedEnds ends{};
    for (int k = kMixedContainers - 1; k >= 0; --k) {
        order[0].insert(order[0].end(), container[k].begin(), container[k].end());
        ends.end[k] = (uint32_t)order[0].size();
    }
    const uint32_t ntiles = (uint32_t)tile_bucket.size(), nmx = ends.end[0];
    const bool both = ntiles && nmx;
    (void)hipSetDevice(e->opt.device);
    pgap_status st;
    hipError_t he;
    // The one-lane kernel runs beside the matrix-core kernel on a stream of
    // its own, created for this call and destroyed at its end: a process
    // gets a few hardware queues (GPU_MAX_HW_QUEUES, 4 by default), and a
    // stream kept alive would make the streaming scan's two streams share
    // one with another (measured: 9.8 k -> 6.7 k m/s at 1511#).
    struct AuxStream {
        hipStream_t s = nullptr;
        hipEvent_t ev = nullptr;
        ~AuxStream() {
            if (s) {
                (void)hipStreamSynchronize(s);
                (void)hipStreamDestroy(s);
            }
            if (ev) (void)hipEventDestroy(ev);
        }
    } aux;
    if (both) {
        if ((he = hipStreamCreateWithFlags(&aux.s, hipStreamNonBlocking)) != hipSuccess ||
            (he = hipEventCreateWithFlags(&aux.ev, hipEventDisableTiming)) != hipSuccess)
            return e->hip_fail(he, "mixed stream");
    }
    const size_t b_words = total_words * 4, b_off = count * 8, b_limbs = count * 4;
    const size_t b_order = (order[0].size() + order[1].size()) * 4;
    if ((st = e->ensure(e->d_n, b_words + b_off + b_limbs + b_order + ntiles + 64, "mixed inputs")) ||
        (st = e->ensure(e->d_out, count, "verdicts")) || (st = e->ensure(e->d_small, 64, "tile counters")))
        return st;
    char *base = (char *)e->d_n.p;
    uint32_t *d_words = (uint32_t *)base;
    uint64_t *d_off = (uint64_t *)(base + ((b_words + 7) & ~(size_t)7));
    uint32_t *d_limbs = (uint32_t *)((char *)d_off + b_off);
    uint32_t *d_order0 = (uint32_t *)((char *)d_limbs + b_limbs);
    uint32_t *d_order1 = d_order0 + order[0].size();
    uint8_t *d_tb = (uint8_t *)(d_order1 + order[1].size());
    uint32_t *d_next = (uint32_t *)e->d_small.p;
    if ((he = hipMemcpyAsync(d_words, words, b_words, hipMemcpyHostToDevice, e->stream)) != hipSuccess ||
        (he = hipMemcpyAsync(d_off, offset, b_off, hipMemcpyHostToDevice, e->stream)) != hipSuccess ||
        (he = hipMemcpyAsync(d_limbs, limbs, b_limbs, hipMemcpyHostToDevice, e->stream)) != hipSuccess ||
        (order[0].size() && (he = hipMemcpyAsync(d_order0, order[0].data(), order[0].size() * 4,
                                                 hipMemcpyHostToDevice, e->stream)) != hipSuccess) ||
        (order[1].size() && (he = hipMemcpyAsync(d_order1, order[1].data(), order[1].size() * 4,
                                                 hipMemcpyHostToDevice, e->stream)) != hipSuccess) ||
        (ntiles && (he = hipMemcpyAsync(d_tb, tile_bucket.data(), ntiles, hipMemcpyHostToDevice, e->stream)) !=
                       hipSuccess) ||
        (he = hipMemsetAsync(d_next, 0, 4, e->stream)) != hipSuccess)
        return e->hip_fail(he, "mixed upload");
    const MixedLaunch mx{d_words, d_off, d_limbs, d_order0, nullptr, 0, nullptr, bs, (uint8_t *)e->d_out.p};
    const MixedLaunch one{d_words, d_off, d_limbs, d_order1, d_tb, ntiles, d_next, bs, (uint8_t *)e->d_out.p};
    // the matrix-core kernel (the widest numbers) on the engine's stream, the
    // one-lane kernel beside it on the second stream; the second joins the
    // first before the end event
    if ((he = hipEventRecord(e->ev0, e->stream)) != hipSuccess) return e->hip_fail(he, "event");
    if (nmx) {
        he = kind == PGAP_FERMAT2 ? launch_mixed_mf_fermat(mx, ends, e->stream)
                                  : launch_mixed_mf_sprp(mx, ends, e->stream);
        if (he != hipSuccess) return e->hip_fail(he, "mixed matrix-core kernel");
    }
    if (ntiles) {
        hipStream_t s1 = both ? aux.s : e->stream;
        if (both && (he = hipStreamWaitEvent(s1, e->ev0, 0)) != hipSuccess) return e->hip_fail(he, "mixed stream");
        he = kind == PGAP_FERMAT2 ? launch_mixed_fermat(one, e->opt.device, s1)
                                  : launch_mixed_sprp(one, e->opt.device, s1);
        if (he != hipSuccess) return e->hip_fail(he, "mixed kernel");
        if (both && ((he = hipEventRecord(aux.ev, s1)) != hipSuccess ||
                     (he = hipStreamWaitEvent(e->stream, aux.ev, 0)) != hipSuccess))
            return e->hip_fail(he, "mixed stream");
    }
    if ((he = hipEventRecord(e->ev1, e->stream)) != hipSuccess) return e->hip_fail(he, "event");
    e->last.digits = 0;
    e->last.radix_bits = 28;
    e->last.lanes_per_number = 0;  // per bucket
    e->last.launches = (uint32_t)((nmx + kMatrixMaxBlocks - 1ull) / kMatrixMaxBlocks) + (ntiles ? 1u : 0u);
    e->last.tests = count;
    e->last.matrix_tests = nmx;
    e->timing_pending = true;
    if ((he = hipMemcpyAsync(verdict, e->d_out.p, count, hipMemcpyDeviceToHost, e->stream)) != hipSuccess ||
        (he = hipStreamSynchronize(e->stream)) != hipSuccess)
        return e->hip_fail(he, "mixed readback");
    e->collect_timing();
    return PGAP_OK;
}
