// silu(g) = bf16(g * sigmoid(g)) for every bf16 gate value g, with each step rounded to bf16 exactly as the
// SwiGLU epilogue computes it (e = bf16(exp|g|), y = bf16(1 / bf16(1 + e)), sigmoid = g < 0 ? y : bf16(1 - y)).
// The rounded sigmoid is 0.5 up to |g| = 2^-8 and the same from |g| = 89 on, so 2048 entries a sign hold all of it and
// the epilogue's ~60 instructions per output become one 2-byte load and a multiplication; the table is evaluated by the
// compiler from the functions below (plain IEEE single-precision operations, the same sequence as swiglu_bf16 / exp_pos
// in scmx_common.h), so it cannot drift from them, and compared with them for every gate value.
#pragma once
#include <cstdint>

namespace scmx {

// Entry of a gate (its bf16 bits): |g| clamped to the 2048 bf16 values from 2^-8 on.
constexpr uint32_t SIGMOID_ENTRIES = 2048, SIGMOID_FIRST = 0x3B80u;
constexpr uint32_t sigmoid_entry(uint32_t gb) {
    const uint32_t a = gb & 0x7FFFu, last = SIGMOID_FIRST + SIGMOID_ENTRIES - 1;
    return (a < SIGMOID_FIRST ? SIGMOID_FIRST : a > last ? last : a) - SIGMOID_FIRST + ((gb >> 15) * SIGMOID_ENTRIES);
}

namespace silu_ce {

constexpr float from_bits(uint32_t u) { return __builtin_bit_cast(float, u); }
constexpr uint32_t to_bits(float f) { return __builtin_bit_cast(uint32_t, f); }
constexpr uint16_t to_bf16(float f) {   // round to nearest even; NaN stays NaN
    uint32_t u = to_bits(f);
    if ((u & 0x7FFFFFFFu) > 0x7F800000u) return uint16_t((u >> 16) | 0x40u);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return uint16_t(u >> 16);
}
constexpr float round_bf16(float f) { return from_bits(uint32_t(to_bf16(f)) << 16); }
constexpr float rint_pos(float x) {   // round half to even for 0 <= x < 2^23
    int i = int(x);
    const float fr = x - float(i);
    if (fr > 0.5f || (fr == 0.5f && (i & 1))) ++i;
    return float(i);
}
constexpr float exp_pos(float a) {
    a = (a < 89.0f) ? a : 89.0f;
    const float n = rint_pos(a * 1.4426950408889634f);
    const float r = (a - n * 0.693145751953125f) - n * 1.428606765330187e-06f;
    float p = 1.0f / 5040.0f;
    p = p * r + 1.0f / 720.0f;
    p = p * r + 1.0f / 120.0f;
    p = p * r + 1.0f / 24.0f;
    p = p * r + 1.0f / 6.0f;
    p = p * r + 0.5f;
    p = p * r + 1.0f;
    p = p * r + 1.0f;
    const int ni = int(n), h = ni >> 1;
    return (p * from_bits(uint32_t(h + 127) << 23)) * from_bits(uint32_t(ni - h + 127) << 23);
}
constexpr uint16_t sigmoid_bits(uint16_t gb) {   // gb: not a NaN
    const float g = from_bits(uint32_t(gb) << 16);
    const float e = round_bf16(exp_pos(g < 0.0f ? -g : g));
    const float y = round_bf16(1.0f / round_bf16(1.0f + e));
    return to_bf16((g < 0.0f) ? y : round_bf16(1.0f - y));
}

struct alignas(16) Table {             // (kernels copy it in pieces of 16 bytes)
    uint16_t v[2 * SIGMOID_ENTRIES];   // of g >= 0, then of g < 0
};
constexpr Table make() {
    Table t{};
    for (uint32_t i = 0; i < 2 * SIGMOID_ENTRIES; ++i)
        t.v[i] = sigmoid_bits(uint16_t(SIGMOID_FIRST + i % SIGMOID_ENTRIES + (i < SIGMOID_ENTRIES ? 0u : 0x8000u)));
    return t;
}
constexpr bool covers_every_gate() {
    const Table t = make();
    for (uint32_t gb = 0; gb < 65536; ++gb)
        if ((gb & 0x7FFFu) <= 0x7F80u && t.v[sigmoid_entry(gb)] != sigmoid_bits(uint16_t(gb))) return false;
    return true;
}
static_assert(covers_every_gate(), "the table's ends stand for the gates beyond them");

}  // namespace silu_ce
}  // namespace scmx
