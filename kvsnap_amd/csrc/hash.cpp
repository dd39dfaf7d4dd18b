// SHA-256 (FIPS 180-4) and CRC32C of records in host memory on host threads,
// with the x86 SHA and CRC32 instructions.
//
// A SHA-256 chain is sequential, so a record's time on the GPU is its chain's
// issue time (0.97 us a 64-byte block) however few records there are, while a
// host core with the SHA extensions runs a chain some 35 times as fast.  A save
// of few records hashes sooner here, from the pinned records it has just
// written; many records hash sooner on the GPU, beside their copies.  Callers
// share the helping threads: all of a process's calls together start no more
// than one of them asked for.
#include "common.h"

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <stdexcept>
#include <thread>
#include <vector>

#if !defined(__HIP_DEVICE_COMPILE__)

#include <cpuid.h>
#include <immintrin.h>

namespace {

bool has_sha_extensions() {
    unsigned a = 0, b = 0, c = 0, d = 0;
    if (!__get_cpuid(1, &a, &b, &c, &d) || !(c & (1u << 9)) || !(c & (1u << 19)) || !(c & (1u << 20))) return false;
    return __get_cpuid_count(7, 0, &a, &b, &c, &d) && (b & (1u << 29));  // SSSE3, SSE4.1, SSE4.2; SHA
}

alignas(16) const uint32_t kRound[64] = {
    0x428a2f98, 0x71374491, 0xb5c0fbcf, 0xe9b5dba5, 0x3956c25b, 0x59f111f1, 0x923f82a4, 0xab1c5ed5,
    0xd807aa98, 0x12835b01, 0x243185be, 0x550c7dc3, 0x72be5d74, 0x80deb1fe, 0x9bdc06a7, 0xc19bf174,
    0xe49b69c1, 0xefbe4786, 0x0fc19dc6, 0x240ca1cc, 0x2de92c6f, 0x4a7484aa, 0x5cb0a9dc, 0x76f988da,
    0x983e5152, 0xa831c66d, 0xb00327c8, 0xbf597fc7, 0xc6e00bf3, 0xd5a79147, 0x06ca6351, 0x14292967,
    0x27b70a85, 0x2e1b2138, 0x4d2c6dfc, 0x53380d13, 0x650a7354, 0x766a0abb, 0x81c2c92e, 0x92722c85,
    0xa2bfe8a1, 0xa81a664b, 0xc24b8b70, 0xc76c51a3, 0xd192e819, 0xd6990624, 0xf40e3585, 0x106aa070,
    0x19a4c116, 0x1e376c08, 0x2748774c, 0x34b0bcb5, 0x391c0cb3, 0x4ed8aa4a, 0x5b9cca4f, 0x682e6ff3,
    0x748f82ee, 0x78a5636f, 0x84c87814, 0x8cc70208, 0x90befffa, 0xa4506ceb, 0xbef9a3f7, 0xc67178f2,
};

#define KVSNAP_SHA_TARGET __attribute__((target("sha,sse4.1,ssse3,sse4.2")))

// One chain: the state as the SHA instructions hold it, (a, b, e, f) and (c, d, g, h) from the high word down.
struct Chain {
    __m128i abef, cdgh;
};

KVSNAP_SHA_TARGET inline Chain chain_start() {
    return Chain{_mm_set_epi32(0x6a09e667, static_cast<int>(0xbb67ae85), 0x510e527f, static_cast<int>(0x9b05688c)),
                 _mm_set_epi32(0x3c6ef372, static_cast<int>(0xa54ff53a), 0x1f83d9ab, 0x5be0cd19)};
}

// kLanes chains through one 64-byte block each.  A chain's rounds wait on each other (sha256rnds2 does two),
// so two chains side by side take little longer than one.
template <int kLanes>
KVSNAP_SHA_TARGET inline void compress(Chain* chain, const uint8_t* const* block) {
    const __m128i swap = _mm_set_epi8(12, 13, 14, 15, 8, 9, 10, 11, 4, 5, 6, 7, 0, 1, 2, 3);
    __m128i w[kLanes][4], abef[kLanes], cdgh[kLanes];
    for (int l = 0; l < kLanes; ++l) {
        abef[l] = chain[l].abef;
        cdgh[l] = chain[l].cdgh;
        for (int i = 0; i < 4; ++i)
            w[l][i] = _mm_shuffle_epi8(_mm_loadu_si128(reinterpret_cast<const __m128i*>(block[l] + 16 * i)), swap);
    }
#pragma GCC unroll 16
    for (int g = 0; g < 16; ++g) {  // rounds 4g .. 4g + 3
        const __m128i k = _mm_load_si128(reinterpret_cast<const __m128i*>(kRound + 4 * g));
        for (int l = 0; l < kLanes; ++l) {
            __m128i* x = w[l];
            if (g >= 4) {  // W[t] from W[t-16], s0(W[t-15]), W[t-7] and s1(W[t-2]), four at a time
                const __m128i first = _mm_sha256msg1_epu32(x[g & 3], x[(g + 1) & 3]);
                const __m128i seventh = _mm_alignr_epi8(x[(g + 3) & 3], x[(g + 2) & 3], 4);
                x[g & 3] = _mm_sha256msg2_epu32(_mm_add_epi32(first, seventh), x[(g + 3) & 3]);
            }
            const __m128i wk = _mm_add_epi32(x[g & 3], k);
            cdgh[l] = _mm_sha256rnds2_epu32(cdgh[l], abef[l], wk);
            abef[l] = _mm_sha256rnds2_epu32(abef[l], cdgh[l], _mm_shuffle_epi32(wk, 0x0E));
        }
    }
    for (int l = 0; l < kLanes; ++l) {
        chain[l].abef = _mm_add_epi32(chain[l].abef, abef[l]);
        chain[l].cdgh = _mm_add_epi32(chain[l].cdgh, cdgh[l]);
    }
}

// kLanes records of `nbytes`: SHA-256 digests and CRC32Cs.  The CRC32C's chain (8 bytes a step) runs in the
// SHA rounds' shadow.
template <int kLanes>
KVSNAP_SHA_TARGET void hash_lanes(const uint8_t* const* records, uint64_t nbytes, uint8_t* const* digests,
                                  uint32_t* const* crcs) {
    Chain chain[kLanes];
    uint64_t crc[kLanes];
    const uint8_t* at[kLanes];
    for (int l = 0; l < kLanes; ++l) {
        chain[l] = chain_start();
        crc[l] = 0xFFFFFFFFu;
        at[l] = records[l];
    }
    const uint64_t whole = nbytes / 64;
    for (uint64_t b = 0; b < whole; ++b) {
        for (int l = 0; l < kLanes; ++l)
            for (int i = 0; i < 8; ++i) {
                uint64_t word;
                std::memcpy(&word, at[l] + 8 * i, 8);
                crc[l] = _mm_crc32_u64(crc[l], word);
            }
        compress<kLanes>(chain, at);
        for (int l = 0; l < kLanes; ++l) at[l] += 64;
    }
    // The padding: 0x80, zeros, the length in bits (big endian), one block or two.
    const uint64_t rest = nbytes - 64 * whole;
    const int final_blocks = rest + 9 <= 64 ? 1 : 2;
    uint8_t tail[kLanes][128] = {};
    for (int l = 0; l < kLanes; ++l) {
        for (uint64_t i = 0; i < rest; ++i) crc[l] = _mm_crc32_u8(static_cast<uint32_t>(crc[l]), at[l][i]);
        std::memcpy(tail[l], at[l], rest);
        tail[l][rest] = 0x80;
        for (int i = 0; i < 8; ++i)
            tail[l][64 * final_blocks - 1 - i] = static_cast<uint8_t>((nbytes * 8) >> (8 * i));
    }
    for (int b = 0; b < final_blocks; ++b) {
        for (int l = 0; l < kLanes; ++l) at[l] = tail[l] + 64 * b;
        compress<kLanes>(chain, at);
    }
    for (int l = 0; l < kLanes; ++l) {
        alignas(16) uint32_t x[4], y[4];  // f, e, b, a and h, g, d, c
        _mm_store_si128(reinterpret_cast<__m128i*>(x), chain[l].abef);
        _mm_store_si128(reinterpret_cast<__m128i*>(y), chain[l].cdgh);
        const uint32_t words[8] = {x[3], x[2], y[3], y[2], x[1], x[0], y[1], y[0]};
        for (int i = 0; i < 8; ++i) {
            const uint32_t big = __builtin_bswap32(words[i]);
            std::memcpy(digests[l] + 4 * i, &big, 4);
        }
        *crcs[l] = ~static_cast<uint32_t>(crc[l]);
    }
}

std::atomic<int> g_helpers{0};  // threads of this process that help a call now

bool take_helper(int most) {
    int now = g_helpers.load(std::memory_order_relaxed);
    while (now < most)
        if (g_helpers.compare_exchange_weak(now, now + 1, std::memory_order_relaxed)) return true;
    return false;
}

void hash_records(const uint64_t* records, uint64_t nbytes, int64_t n, uint8_t* digests, uint32_t* crcs, int threads) {
    // A thread is worth starting (about 15 us) for 64 KiB of its own, and has one record or, where there are more
    // records than threads, pairs of them; it takes the next when it is done with its last.
    const int64_t pairs = (n + 1) / 2;
    const int64_t useful = std::min<int64_t>({threads, n > threads ? pairs : n, static_cast<int64_t>(nbytes * n >> 16)});
    int64_t helpers = 0;
    while (helpers + 1 < useful && take_helper(threads - 1)) ++helpers;
    const int64_t lanes = n > helpers + 1 ? 2 : 1, jobs = (n + lanes - 1) / lanes;
    std::atomic<int64_t> next{0};
    const auto work = [&] {
        for (int64_t job; (job = next.fetch_add(1, std::memory_order_relaxed)) < jobs;) {
            const int64_t first = job * lanes;
            const uint8_t* in[2];
            uint8_t* sha[2];
            uint32_t* crc[2];
            const int64_t count = std::min<int64_t>(lanes, n - first);
            for (int64_t l = 0; l < count; ++l) {
                in[l] = reinterpret_cast<const uint8_t*>(records[first + l]);
                sha[l] = digests + 32 * (first + l);
                crc[l] = crcs + first + l;
            }
            if (count == 2)
                hash_lanes<2>(in, nbytes, sha, crc);
            else
                hash_lanes<1>(in, nbytes, sha, crc);
        }
    };
    std::vector<std::thread> others;
    int64_t untaken = helpers;
    try {
        others.reserve(static_cast<size_t>(helpers));
        for (; untaken > 0; --untaken)
            others.emplace_back([&work] {
                work();
                g_helpers.fetch_sub(1, std::memory_order_relaxed);
            });
    } catch (...) {
        // No more threads to be had: the ones there are, this one at least, do all the work.
        g_helpers.fetch_sub(static_cast<int>(untaken), std::memory_order_relaxed);
    }
    work();
    for (auto& thread : others) thread.join();
}

}  // namespace

extern "C" {

int kvsnap_hash_records_available() { return has_sha_extensions() ? 1 : 0; }

int kvsnap_hash_records(const uint64_t* records, uint64_t record_bytes, int64_t n_records, uint8_t* digests,
                        uint32_t* crcs, int threads) {
    try {
        if (n_records < 0 || threads < 1 || threads > 256)
            throw std::runtime_error("host hashes: a record count and 1 to 256 threads");
        if (n_records == 0) return 0;
        if (!records || !digests || !crcs) throw std::runtime_error("host hashes need records and outputs");
        if (record_bytes > (uint64_t(1) << 40) / static_cast<uint64_t>(n_records))
            throw std::runtime_error("host hashes: at most 1 TiB a call");
        if (!has_sha_extensions()) throw std::runtime_error("host hashes need the SHA and SSE4.2 instructions");
        hash_records(records, record_bytes, n_records, digests, crcs, threads);
        return 0;
    } catch (const std::exception& e) {
        kvsnap::set_error(e.what());
        return -1;
    }
}

}  // extern "C"

#endif  // !__HIP_DEVICE_COMPILE__
