// LDS strides of the y-z kernels with the fewest bank conflicts (written by
// gen_yz_pads.py, which says how they are chosen).
#pragma once

namespace amdk {

// bytes: sizeof of a complex value (8 or 16)
template <int N, int bytes> struct YzPads;
template <> struct YzPads<20, 8> { static constexpr int PS = 37, RS = 4, CS = 47, RX = 6, RY = 6; };
template <> struct YzPads<20, 16> { static constexpr int PS = 21, RS = 4, CS = 25, RX = 5, RY = 5; };
template <> struct YzPads<24, 8> { static constexpr int PS = 27, RS = 4, CS = 58, RX = 4, RY = 7; };
template <> struct YzPads<24, 16> { static constexpr int PS = 27, RS = 4, CS = 36, RX = 5, RY = 7; };
template <> struct YzPads<30, 8> { static constexpr int PS = 37, RS = 6, CS = 35, RX = 5, RY = 7; };
template <> struct YzPads<30, 16> { static constexpr int PS = 30, RS = 5, CS = 35, RX = 5, RY = 7; };
template <> struct YzPads<32, 8> { static constexpr int PS = 40, RS = 5, CS = 40, RX = 5, RY = 9; };
template <> struct YzPads<32, 16> { static constexpr int PS = 38, RS = 4, CS = 37, RX = 4, RY = 8; };
template <> struct YzPads<36, 8> { static constexpr int PS = 59, RS = 7, CS = 39, RX = 6, RY = 6; };
template <> struct YzPads<36, 16> { static constexpr int PS = 42, RS = 7, CS = 42, RX = 7, RY = 7; };
template <> struct YzPads<40, 8> { static constexpr int PS = 40, RS = 5, CS = 56, RX = 5, RY = 9; };
template <> struct YzPads<40, 16> { static constexpr int PS = 41, RS = 5, CS = 41, RX = 5, RY = 8; };
template <> struct YzPads<48, 8> { static constexpr int PS = 56, RS = 7, CS = 56, RX = 7, RY = 9; };
template <> struct YzPads<48, 16> { static constexpr int PS = 54, RS = 6, CS = 49, RX = 6, RY = 8; };
template <> struct YzPads<50, 8> { static constexpr int PS = 55, RS = 5, CS = 50, RX = 5, RY = 10; };
template <> struct YzPads<50, 16> { static constexpr int PS = 58, RS = 5, CS = 55, RX = 5, RY = 10; };
template <> struct YzPads<54, 8> { static constexpr int PS = 57, RS = 6, CS = 70, RX = 7, RY = 11; };
template <> struct YzPads<54, 16> { static constexpr int PS = 57, RS = 6, CS = 56, RX = 6, RY = 9; };
template <> struct YzPads<60, 8> { static constexpr int PS = 70, RS = 7, CS = 70, RX = 7, RY = 11; };
template <> struct YzPads<60, 16> { static constexpr int PS = 61, RS = 6, CS = 61, RX = 6, RY = 10; };
template <> struct YzPads<64, 8> { static constexpr int PS = 72, RS = 9, CS = 72, RX = 9, RY = 9; };
template <> struct YzPads<64, 16> { static constexpr int PS = 72, RS = 9, CS = 72, RX = 9, RY = 9; };
template <> struct YzPads<72, 8> { static constexpr int PS = 73, RS = 8, CS = 81, RX = 9, RY = 9; };
template <> struct YzPads<72, 16> { static constexpr int PS = 73, RS = 8, CS = 81, RX = 9, RY = 9; };
template <> struct YzPads<80, 8> { static constexpr int PS = 90, RS = 9, CS = 119, RX = 10, RY = 10; };
template <> struct YzPads<80, 16> { static constexpr int PS = 90, RS = 9, CS = 104, RX = 9, RY = 11; };
template <> struct YzPads<90, 8> { static constexpr int PS = 90, RS = 9, CS = 105, RX = 10, RY = 10; };
template <> struct YzPads<90, 16> { static constexpr int PS = 90, RS = 9, CS = 110, RX = 11, RY = 11; };
template <> struct YzPads<96, 8> { static constexpr int PS = 97, RS = 8, CS = 97, RX = 8, RY = 12; };
template <> struct YzPads<96, 16> { static constexpr int PS = 121, RS = 9, CS = 108, RX = 9, RY = 13; };
template <> struct YzPads<100, 8> { static constexpr int PS = 110, RS = 11, CS = 105, RX = 10, RY = 10; };
template <> struct YzPads<100, 16> { static constexpr int PS = 122, RS = 11, CS = 110, RX = 11, RY = 11; };
template <> struct YzPads<108, 8> { static constexpr int PS = 108, RS = 9, CS = 117, RX = 9, RY = 13; };
template <> struct YzPads<108, 16> { static constexpr int PS = 121, RS = 9, CS = 117, RX = 9, RY = 13; };
template <> struct YzPads<120, 8> { static constexpr int PS = 121, RS = 10, CS = 133, RX = 11, RY = 13; };
template <> struct YzPads<120, 16> { static constexpr int PS = 123, RS = 10, CS = 121, RX = 10, RY = 12; };
template <> struct YzPads<128, 8> { static constexpr int PS = 146, RS = 9, CS = 144, RX = 9, RY = 17; };
template <> struct YzPads<128, 16> { static constexpr int PS = 129, RS = 8, CS = 129, RX = 8, RY = 16; };
template <> struct YzPads<144, 8> { static constexpr int PS = 172, RS = 13, CS = 156, RX = 13, RY = 13; };
template <> struct YzPads<144, 16> { static constexpr int PS = 145, RS = 12, CS = 145, RX = 12, RY = 12; };
template <> struct YzPads<150, 8> { static constexpr int PS = 175, RS = 11, CS = 176, RX = 11, RY = 15; };
template <> struct YzPads<150, 16> { static constexpr int PS = 151, RS = 10, CS = 151, RX = 10, RY = 15; };
template <> struct YzPads<160, 8> { static constexpr int PS = 170, RS = 10, CS = 176, RX = 11, RY = 17; };
template <> struct YzPads<160, 16> { static constexpr int PS = 161, RS = 10, CS = 161, RX = 10, RY = 16; };
template <> struct YzPads<162, 8> { static constexpr int PS = 182, RS = 19, CS = 171, RX = 18, RY = 9; };
template <> struct YzPads<162, 16> { static constexpr int PS = 163, RS = 18, CS = 163, RX = 18, RY = 9; };
template <> struct YzPads<180, 8> { static constexpr int PS = 182, RS = 12, CS = 208, RX = 13, RY = 15; };
template <> struct YzPads<180, 16> { static constexpr int PS = 181, RS = 12, CS = 181, RX = 12, RY = 15; };
template <> struct YzPads<192, 8> { static constexpr int PS = 193, RS = 12, CS = 193, RX = 12, RY = 16; };
template <> struct YzPads<192, 16> { static constexpr int PS = 193, RS = 12, CS = 193, RX = 12, RY = 16; };

}  // namespace amdk
