// 64-bit content fingerprint of host byte ranges: tells apart scenes, material tables, envmaps
// and checkpoint payloads. Not cryptographic; it catches a snapshot resumed into another
// scene and bytes changed in storage.
#pragma once
#include <stddef.h>
#include <stdint.h>

#include <cstring>

namespace rgpu {

inline uint64_t fp_mix(uint64_t h) {  // the splitmix64 finaliser
    h ^= h >> 30;
    h *= 0xbf58476d1ce4e5b9ull;
    h ^= h >> 27;
    h *= 0x94d049bb133111ebull;
    h ^= h >> 31;
    return h;
}

// Four independent multiply-rotate lanes over 32-byte blocks (so the loop runs near memory
// speed), folded with the length and the tail at the end. Bytes may come in pieces; every piece
// but the last is a multiple of 32 bytes.
struct Fingerprint {
    uint64_t a, b, c, d;
    uint64_t bytes = 0;
    uint8_t tail[32];
    size_t ntail = 0;
    explicit Fingerprint(uint64_t seed = 0)
        : a(seed ^ 0x243f6a8885a308d3ull), b(seed ^ 0x13198a2e03707344ull), c(seed ^ 0xa4093822299f31d0ull),
          d(seed ^ 0x082efa98ec4e6c89ull) {}
    void add(const void* data, size_t n) {
        const uint8_t* p = static_cast<const uint8_t*>(data);
        const uint64_t k = 0x9e3779b97f4a7c15ull;
        uint64_t x = a, y = b, z = c, v = d;
        size_t i = 0;
        for (; i + 32 <= n; i += 32) {
            uint64_t w[4];
            std::memcpy(w, p + i, 32);
            x = ((x ^ w[0]) * k);
            x = (x << 29) | (x >> 35);
            y = ((y ^ w[1]) * k);
            y = (y << 29) | (y >> 35);
            z = ((z ^ w[2]) * k);
            z = (z << 29) | (z >> 35);
            v = ((v ^ w[3]) * k);
            v = (v << 29) | (v >> 35);
        }
        a = x;
        b = y;
        c = z;
        d = v;
        bytes += n;
        ntail = n - i;
        std::memcpy(tail, p + i, ntail);
    }
    uint64_t value() const {
        const uint64_t k = 0x9e3779b97f4a7c15ull;
        uint64_t h = fp_mix(a) ^ fp_mix(b + 1) ^ fp_mix(c + 2) ^ fp_mix(d + 3) ^ fp_mix(bytes + k);
        for (size_t j = 0; j < ntail; ++j) h = fp_mix(h ^ (uint64_t)tail[j] ^ ((bytes - ntail + j) << 8));
        return fp_mix(h);
    }
};

inline uint64_t fingerprint64(const void* data, size_t bytes, uint64_t seed = 0) {
    Fingerprint f(seed);
    if (bytes) f.add(data, bytes);
    return f.value();
}

}  // namespace rgpu
