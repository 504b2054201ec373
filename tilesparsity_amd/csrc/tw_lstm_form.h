// Which of its two kernels a multi-step LSTM launch takes.
#ifndef TW_LSTM_FORM_H
#define TW_LSTM_FORM_H

#include <cstdint>

namespace tw {

constexpr int kPanRows = 1024; // most rows of x, and of h, that the form with the rows of A in LDS keeps there

// The form with the rows of A in LDS, for tiles of `kept` rows in the mean.  It saves up to a fifth of a step and needs 4 - 6 us more to begin with.  us for
// 50 steps, the other form and in LDS, inputs as many as units: H 1024, a quarter kept, M 8 204 and 182, M 128 228 and 200, M 200 275 and 228, M 256 225 and 211;
// a tenth M 8 182 and 154, M 128 194 and 159; M 1 a quarter 201 and 195, a tenth 168 and 163; H 512, a quarter, M 128 176 and 158, half 210 and 178, a tenth 147
// and 146; H 256 138 and 145.  24 steps: H 1024, 512 inputs, 154 kept rows, M 2 91 and 85, M 128 97 and 85; 64 inputs, 109 kept 79 and 83.  Below H 1024 with few
// rows or few kept rows of h: H 512, 1024 inputs, M 16, 102 of h 77 and 84, M 128, 51 of h 79 and 78; H 768, 768 inputs, M 4, 154 of h 90 and 94.
inline bool lstm_rows_in_lds(int K, int H, int M, int T, int64_t kept)
{
    return K > H && K - H <= kPanRows && H <= kPanRows && M >= 2 && kept >= 150 &&
           (H >= 1024 ? T >= 24 : H >= 512 && T >= 32 && M > 32 && kept * H >= 100 * (int64_t)K);
}

} // namespace tw
#endif
