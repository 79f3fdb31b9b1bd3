// Generated by gen_obc_farfield.py -- do not edit by hand.
// Far-field OBC2 pair integral polynomials in y = (s/r)^2 on [0, 0.25].
// max relative error: h 3.01e-08, k 1.23e-08
#pragma once
#define PRX_OBC_FAR_YMAX 0.25f
#define PRX_OBC_FAR_XMAX 0.5f
constexpr int kObcHDeg = 6;
__device__ constexpr float kObcH[7] = {0.66666668674528928f, 0.79999229003459049f, 0.85762308360337824f, 0.8777862666882047f, 1.029180855970844f, 0.27933811005615627f, 2.4965702391961209f};
constexpr int kObcKDeg = 7;
__device__ constexpr float kObcK[8] = {1.3333333168974937f, 2.400008251869155f, 3.4278952757724479f, 4.4653877565721238f, 5.1398458343982405f, 8.9759534420397742f, -3.2064037352076404f, 29.639321640249108f};
// The same on [0, 0.0625] (s <= r/4); max relative error: h 3.08e-09, k 1.11e-08
#define PRX_OBC_FAR4_YMAX 0.0625f
#define PRX_OBC_FAR4_XMAX 0.25f
constexpr int kObcH4Deg = 4;
__device__ constexpr float kObcH4[5] = {0.66666666872154989f, 0.79999836766752519f, 0.85734960136170812f, 0.87978772663299587f, 1.0697785612734509f};
constexpr int kObcK4Deg = 4;
__device__ constexpr float kObcK4[5] = {1.3333333480933838f, 2.3999882868211322f, 3.4300527588646554f, 4.3793952777570881f, 6.5973534742035334f};
// The same for s <= r/6.5; max relative error: h 3.53e-09, k 1.07e-08
#define PRX_OBC_FAR3_XMAX 0.153846154f
constexpr int kObcH3Deg = 3, kObcK3Deg = 3;
__device__ constexpr float kObcH3[4] = {0.66666666431269472f, 0.80000317176590752f, 0.85647660317730745f, 0.93342088098950193f};
__device__ constexpr float kObcK3[4] = {1.3333333190797376f, 2.4000191945887033f, 3.4245432458952312f, 4.7131794432933019f};
// The same for s <= r/14.5; max relative error: h 4.52e-09, k 1.13e-08
#define PRX_OBC_FAR2_XMAX 0.0689655172f
constexpr int kObcH2Deg = 2, kObcK2Deg = 2;
__device__ constexpr float kObcH2[3] = {0.66666666968101695f, 0.79998860299052732f, 0.86352069034728762f};
__device__ constexpr float kObcK2[3] = {1.3333333484308443f, 2.399942928361444f, 3.460496959115233f};
