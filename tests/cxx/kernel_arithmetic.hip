// The kernels' shortened exponential and division (csrc/common.hpp), compiled for the host, against what they stand for.
// Each part prints how many of its inputs differ; the exit code says whether any does that must not.
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <atomic>
#include <functional>
#include <random>
#include <thread>
#include <type_traits>
#include <vector>

#include "linear.hpp"

// the factor of a row belongs to grouped products: other kernels do not apply it, so no other epilogue can carry it
template <class EP, class = void>
constexpr bool has_row_scale = false;
template <class EP>
constexpr bool has_row_scale<EP, std::void_t<decltype(EP::row_scale)>> = true;
static_assert(has_row_scale<lcu::linear_epilogue<true, true>> && !has_row_scale<lcu::linear_epilogue<false, true>> &&
              !has_row_scale<lcu::linear_epilogue<false, false>>);

namespace {

float of_bits(uint32_t u) { return __builtin_bit_cast(float, u); }
uint32_t bits(float f) { return __builtin_bit_cast(uint32_t, f); }
uint16_t half_bits(float f) { return __builtin_bit_cast(uint16_t, (_Float16)f); }

// f(first, last) over pieces of [0, n); the sum of what it returns
long in_pieces(uint64_t n, const std::function<long(uint64_t, uint64_t)>& f) {
  std::atomic<uint64_t> next{0};
  std::atomic<long> sum{0};
  std::vector<std::thread> threads;
  const uint64_t piece = n / 256 + 1;
  for (int t = 0; t < 8; ++t) {
    threads.emplace_back([&] {
      for (uint64_t at; (at = next.fetch_add(piece)) < n;) sum += f(at, at + piece < n ? at + piece : n);
    });
  }
  for (auto& t : threads) t.join();
  return sum;
}

int failed = 0;
void report(const char* what, long differ) {
  printf("%s: %ld differ\n", what, differ);
  failed |= differ != 0;
}

}  // namespace

int main() {
  // the exponential: every float in [-104, -0], steps of 16 values from there to -infinity, and NaN
  const uint32_t far = bits(-104.0f), low = bits(-INFINITY);
  report("exp of all x in [-104, 0]", in_pieces(far - 0x80000000u + 1, [](uint64_t a, uint64_t b) {
           long n = 0;
           for (uint64_t i = a; i < b; ++i) {
             const float x = of_bits(0x80000000u + (uint32_t)i);
             n += bits(lcu::exp_ieee(x)) != bits(lcu::exp_ieee_nonpositive(x));
           }
           return n;
         }));
  long rest = lcu::exp_ieee_nonpositive(0.0f) != 1.0f || !isnan(lcu::exp_ieee_nonpositive(NAN));
  for (uint64_t u = far; u <= low; u += 16) rest += lcu::exp_ieee_nonpositive(of_bits((uint32_t)u)) != 0.0f;
  report("exp below", rest + (lcu::exp_ieee_nonpositive(-INFINITY) != 0.0f));

  // scores: every finite x over sqrt(128) (the operation is odd in x)
  const float denom = sqrtf(128.0f), inverse = 1.0f / denom;
  std::atomic<long> small{0};
  report("x / sqrt(128), fp16, or fp32 for x of 2^-100 and more", in_pieces(0x7f800000u, [&](uint64_t a, uint64_t b) {
           long n = 0, s = 0;
           for (uint64_t i = a; i < b; ++i) {
             const float x = of_bits((uint32_t)i), want = x / denom, got = lcu::divide_by(x, denom, inverse);
             if (bits(got) == bits(want)) continue;
             ++s;
             n += x >= 0x1p-100f || half_bits(got) != half_bits(want);
           }
           small += s;
           return n;
         }));
  printf("  (%ld smaller ones differ in fp32)\n", small.load());

  // the same in two instructions, which is for halves only: every float but NaN; and the exponential whose power of two is added to its exponent
  report("score_of, fp16", in_pieces(1ull << 32, [&](uint64_t a, uint64_t b) {
           long n = 0;
           for (uint64_t i = a; i < b; ++i) {
             const float x = of_bits((uint32_t)i);
             n += x == x && half_bits(lcu::score_of(x)) != half_bits(x / denom);
           }
           return n;
         }));
  report("exp of all x in [EXP_LEAST, 0] by its exponent", in_pieces((bits(lcu::EXP_LEAST) - 0x80000000u) / 4 + 1, [](uint64_t a, uint64_t b) {
           long n = 0;
           for (uint64_t i = a; i < b; ++i) {
             float x[4], e[4];
             for (uint32_t k = 0; k < 4; ++k) x[k] = fmaxf(of_bits(0x80000000u + 4 * (uint32_t)i + k), lcu::EXP_LEAST);
             lcu::exp_ieee_above(e, x);
             for (int k = 0; k < 4; ++k) n += bits(e[k]) != bits(lcu::exp_ieee_nonpositive(x[k])) || e[k] < 1e-38f;
           }
           return n;
         }));

  // the quantiser: every pair of a normal fp16 scale and an fp16 value with a quotient of up to 300
  report("halves over fp16 scales", in_pieces(0x7c00 - 0x0400, [](uint64_t a, uint64_t b) {
           long n = 0;
           for (uint64_t i = a; i < b; ++i) {
             const float s = (float)__builtin_bit_cast(_Float16, (uint16_t)(0x0400 + i)), inverse = 1.0f / s;
             for (uint32_t h = 0; h < 0x7c00; ++h) {
               const float x = (float)__builtin_bit_cast(_Float16, (uint16_t)h), want = x / s;
               if (want > 300.0f) break;
               n += bits(lcu::divide_by(x, s, inverse)) != bits(want);
             }
           }
           return n;
         }));

  // logits: every half over temperatures of all sizes (0 of either sign), and probabilities over the sums of a vocabulary
  report("halves over temperatures", in_pieces(4096, [](uint64_t a, uint64_t b) {
           long n = 0;
           for (uint64_t t = a; t < b; ++t) {
             std::mt19937 random((uint32_t)t);
             float d = of_bits(((127 - 40 + random() % 80) << 23) + (t % 3 == 0 ? random() % 64 : t % 3 == 1 ? 0x7fffffu - random() % 64 : random() % (1u << 23)));
             const float usual[4] = {0.8f, 1.0f, 0.1f, 1.5f};
             if (t < 4) d = usual[t];
             if (t % 7 == 6) d = -d;
             const float inverse = 1.0f / d;
             for (uint32_t h = 0; h < 0x10000; ++h) {
               const float x = (float)__builtin_bit_cast(_Float16, (uint16_t)h), want = x / d, got = lcu::divide_rounded(x, d, inverse);
               n += x == x ? got != want : got == got;
             }
           }
           return n;
         }));
  report("samples of e / sum in [1, 32768], fp32 for e of 2^-100 and more, or fp16", in_pieces(4096, [](uint64_t a, uint64_t b) {
           long n = 0;
           for (uint64_t t = a; t < b; ++t) {
             std::mt19937 random((uint32_t)t + 5);
             const float s = of_bits(0x3f800000u + random() % (15u << 23)), share = 1.0f / s;
             for (int i = 0; i < 50000; ++i) {
               const float e = i == 0 ? 0.0f : of_bits(0x00800000u + random() % (0x3f800001u - 0x00800000u));
               const float want = e / s, got = lcu::divide_rounded(e, s, share);
               n += bits(got) != bits(want) && (e >= 0x1p-100f || half_bits(got) != half_bits(want));
             }
           }
           return n;
         }));

  // probabilities: exponentials (0 and 2^-126 .. 1) over sums in [1, 4096], with significands at both ends among the sums
  report("samples of e / sum, fp16, or fp32 for e of 2^-100 and more", in_pieces(4096, [](uint64_t a, uint64_t b) {
           long n = 0;
           for (uint64_t t = a; t < b; ++t) {
             std::mt19937 random((uint32_t)t);
             float s = of_bits(0x3f800000u + random() % (12u << 23));
             if (t < 400) s = of_bits((bits(s) & 0xff800000u) | (t < 200 ? (uint32_t)t : 0x7fffffu - (uint32_t)(t - 200)));
             const float share = 1.0f / s;
             for (int i = 0; i < 50000; ++i) {
               const float e = i == 0 ? 0.0f : of_bits(0x00800000u + random() % (0x3f800001u - 0x00800000u));
               const float want = e / s, got = lcu::divide_by(e, s, share);
               n += bits(got) != bits(want) && (e >= 0x1p-100f || half_bits(got) != half_bits(want));
             }
           }
           return n;
         }));
  return failed;
}
