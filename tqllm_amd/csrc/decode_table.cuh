// Sixteen-entry byte tables looked up with two v_perm_b32 and one exclusive or.
//
// v_perm_b32 with selector bytes 0..7 picks from an eight-byte pool; selectors 8..11 give 0x00 or 0xFF by the sign of pool
// bytes 1, 3, 5 and 7, 12 gives 0x00 and 13..15 give 0xFF. So pool A under the code c and pool B under c ^ 8 each give one
// of their entries for one half of the codes and a known constant for the other half: with the other pool's constant folded
// into the entries (entry ^ constant) the exclusive or of the two picks is the value. The constants depend on the sign bits
// of odd entries of the other pool; taken in the order below every entry depends on entries already known. Eleven
// instructions for eight codes; picking from both halves of the table and then between the picks takes thirteen.
#pragma once
#include "common.cuh"

namespace tqmoe {
namespace {

struct Table16 { uint32_t a0, a1, b0, b1; };
constexpr Table16 table16(const int (&t)[16]) {
    uint32_t a[8] = {}, b[8] = {};
    auto neg = [](uint32_t v) { return (v & 0x80u) ? 0xFFu : 0u; };
    auto val = [&](int i) { return uint32_t(t[i]) & 0xFFu; };
    a[5] = val(5) ^ 0xFFu; a[6] = val(6) ^ 0xFFu; a[7] = val(7) ^ 0xFFu; a[4] = val(4);   // c = 4: selector 12 of pool B, 5..7: 13..15
    b[5] = val(13) ^ 0xFFu; b[6] = val(14) ^ 0xFFu; b[7] = val(15) ^ 0xFFu; b[4] = val(12);
    b[3] = val(11) ^ neg(a[7]); b[2] = val(10) ^ neg(a[5]);                             // codes 8..11: selectors 8..11 of pool A
    a[3] = val(3) ^ neg(b[7]); a[2] = val(2) ^ neg(b[5]); a[1] = val(1) ^ neg(b[3]);
    b[1] = val(9) ^ neg(a[3]); b[0] = val(8) ^ neg(a[1]);
    a[0] = val(0) ^ neg(b[1]);
    auto word = [](const uint32_t * v) { return v[0] | v[1] << 8 | v[2] << 16 | v[3] << 24; };
    return Table16{word(a), word(a + 4), word(b), word(b + 4)};
}
__device__ __forceinline__ uint32_t pick(const Table16 & t, uint32_t c) {   // four codes, one per byte
    return __builtin_amdgcn_perm(t.a1, t.a0, c) ^ __builtin_amdgcn_perm(t.b1, t.b0, c ^ 0x08080808u);
}

}  // namespace
}  // namespace tqmoe
