// erf_exp.h -- exp(-x*x) and erf(x) of one argument in FP64, together.
//
// Every split flux needs both for the same argument (split_fluxes.f90), and
// the library's two routines were half of the FP64 flux kernel's arithmetic.
// Here they come from the nearest of 385 nodes x_j = j/64 and the step
// d = x - x_j, |d| <= 1/128, with p = -2 x_j d and s = d*d:
//   exp(-x*x) = exp(-x_j^2) * exp(p - s)
//   erf(x)    = erf(x_j) + 2/sqrt(pi) * exp(-x_j^2) * integral_0^d exp(-2 x_j t - t^2) dt
//   integral  = d * (A0 - s A1 + s^2/2 A2 - s^3/6 A3),  A_m(p) = sum_n p^n / (n! (n + 2m + 1))
// (expand exp(-t^2) and integrate term by term); exp(p) - 1 = p A0.  The series
// are cut where what is left is below 2e-17 of the results.  d is exact, and
// the node values are rounded once: over |x| <= 6 the largest errors, against
// 200-bit arithmetic, are 1.4 ulp for exp(-x*x) (32 when x*x is rounded
// before the exponential) and 1.1e-16, or 1.5 ulp, for erf.  Beyond
// 6 erf rounds to 1 and exp is taken by itself.  About 40 instructions instead
// of some 120.
#pragma once

#include <hip/hip_runtime.h>

namespace mfcfd {

constexpr int kErfNodes = 385;
// erf(x_j), exp(-x_j*x_j), each the nearest double
static __device__ const double kErfTable[kErfNodes][2] = {
    {0x0.0p+0, 0x1.0000000000000p+0},
    {0x1.20d77083f17a0p-6, 0x1.ffe000fffaaacp-1},
    {0x1.20c5645dd2538p-5, 0x1.ff800ffeaac00p-1},
    {0x1.b0fafef135745p-5, 0x1.fee050f0d2228p-1},
    {0x1.207d480e90658p-4, 0x1.fe00ffaabffbcp-1},
    {0x1.68591a1e83b5dp-4, 0x1.fce26fbaf9ab1p-1},
    {0x1.b0081148a873ap-4, 0x1.fb850c3621ca5p-1},
    {0x1.f78159ec8bb50p-4, 0x1.f9e957744abfap-1},
    {0x1.1f5e1a35c3b89p-3, 0x1.f80feabfeefa5p-1},
    {0x1.42d7fc2f64959p-3, 0x1.f5f975f6d55dap-1},
    {0x1.662a0bdf7a89fp-3, 0x1.f3a6bf1d3472ep-1},
    {0x1.895010fdbdbfdp-3, 0x1.f118a1e372b49p-1},
    {0x1.ac45e37fe2526p-3, 0x1.ee500f1eed967p-1},
    {0x1.cf076d1233237p-3, 0x1.eb4e0c363bc9fp-1},
    {0x1.f190aa85540e2p-3, 0x1.e813b2816996cp-1},
    {0x1.09eed6982b948p-2, 0x1.e4a22e9eb7f0cp-1},
    {0x1.1af54e232d609p-2, 0x1.e0fabfbc702a4p-1},
    {0x1.2bd9db0f7827fp-2, 0x1.dd1eb6d866baap-1},
    {0x1.3c9aa8b84bedap-2, 0x1.d90f75f5cf834p-1},
    {0x1.4d35ef3e5372ep-2, 0x1.d4ce6f4a0d39dp-1},
    {0x1.5da9f415ff23fp-2, 0x1.d05d24612c2afp-1},
    {0x1.6df50a8dff772p-2, 0x1.cbbd253abe533p-1},
    {0x1.7e15944d9d3e4p-2, 0x1.c6f00f5fd3d7fp-1},
    {0x1.8e0a01cab516bp-2, 0x1.c1f78cf2cf2d7p-1},
    {0x1.9dd0d2b721f39p-2, 0x1.bcd553b9d7b62p-1},
    {0x1.ad68966569a87p-2, 0x1.b78b2424b0563p-1},
    {0x1.bccfec24855b8p-2, 0x1.b21ac84eb95f8p-1},
    {0x1.cc058392a6d2dp-2, 0x1.ac8612fde6531p-1},
    {0x1.db081ce6e2a48p-2, 0x1.a6cede9f70468p-1},
    {0x1.e9d68931ae650p-2, 0x1.a0f70c430d437p-1},
    {0x1.f86faa9428f9dp-2, 0x1.9b00829573ba7p-1},
    {0x1.03693a371519cp-1, 0x1.94ed2cdaef21fp-1},
    {0x1.0a7ef5c18edd2p-1, 0x1.8ebef9eac820bp-1},
    {0x1.1178930ada115p-1, 0x1.8877db2c3f2d1p-1},
    {0x1.1855a5fd3dd50p-1, 0x1.8219c395d4690p-1},
    {0x1.1f15cb50bc4dep-1, 0x1.7ba6a6af92b36p-1},
    {0x1.25b8a88b6dd7fp-1, 0x1.752077990e79dp-1},
    {0x1.2c3debfd7d6c1p-1, 0x1.6e892813c2cc1p-1},
    {0x1.32a54cb8db67bp-1, 0x1.67e2a792709adp-1},
    {0x1.38ee8a84beb71p-1, 0x1.612ee24e1cecfp-1},
    {0x1.3f196dcd0f135p-1, 0x1.5a6fc061433c8p-1},
    {0x1.4525c78dd5966p-1, 0x1.53a724e9c91e6p-1},
    {0x1.4b13713ad3513p-1, 0x1.4cd6ed3237e90p-1},
    {0x1.50e24ca35fd2cp-1, 0x1.4600efe2b83d4p-1},
    {0x1.569243d2b3a9bp-1, 0x1.3f26fc3a423a1p-1},
    {0x1.5c2348ecc4dc3p-1, 0x1.384ad9506bc24p-1},
    {0x1.61955607dd15dp-1, 0x1.316e456034a07p-1},
    {0x1.66e86d0312e82p-1, 0x1.2a92f51c26944p-1},
    {0x1.6c1c9759d0e5fp-1, 0x1.23ba930c1568bp-1},
    {0x1.7131e5f496a5ap-1, 0x1.1ce6bef4c13d5p-1},
    {0x1.762870f720c6fp-1, 0x1.16190d4993258p-1},
    {0x1.7b00578c26037p-1, 0x1.0f5306a8a23fdp-1},
    {0x1.7fb9bfaed8078p-1, 0x1.089627612572fp-1},
    {0x1.8454d5f25760dp-1, 0x1.01e3df046c203p-1},
    {0x1.88d1cd474a2e0p-1, 0x1.f67b2002dcc38p-2},
    {0x1.8d30debfc572ep-1, 0x1.e9491e95f7b9cp-2},
    {0x1.91724951b8fc6p-1, 0x1.dc3448110daaep-2},
    {0x1.959651980da31p-1, 0x1.cf3f0ea300349p-2},
    {0x1.999d4192a5715p-1, 0x1.c26bc7e65f17ap-2},
    {0x1.9d8768656cc42p-1, 0x1.b5bcac81d8fbep-2},
    {0x1.a1551a16aaeafp-1, 0x1.a933d7dd220fcp-2},
    {0x1.a506af4cc00f4p-1, 0x1.9cd347e9f70d9p-2},
    {0x1.a89c850b7d54dp-1, 0x1.909cdd00d4565p-2},
    {0x1.ac16fc7143263p-1, 0x1.849259d0eacd1p-2},
    {0x1.af767a741088bp-1, 0x1.78b56362cef38p-2},
    {0x1.b2bb679ead19cp-1, 0x1.6d07812d52816p-2},
    {0x1.b5e62fce16095p-1, 0x1.618a1d3bed529p-2},
    {0x1.b8f741ef54f83p-1, 0x1.563e8466101dap-2},
    {0x1.bbef0fbde6221p-1, 0x1.4b25e696b1e9fp-2},
    {0x1.bece0d82d1a5cp-1, 0x1.4041572360bdfp-2},
    {0x1.c194b1d49a184p-1, 0x1.3591cd321674dp-2},
    {0x1.c443755820d64p-1, 0x1.2b18242d0c1d7p-2},
    {0x1.c6dad2829ec62p-1, 0x1.20d51c43c0ae6p-2},
    {0x1.c95b455cce69dp-1, 0x1.16c95af8633b6p-2},
    {0x1.cbc54b476248dp-1, 0x1.0cf56bb8cd2ecp-2},
    {0x1.ce1962c0e0d8bp-1, 0x1.0359c082364c1p-2},
    {0x1.d0580b2cfd249p-1, 0x1.f3ed651d94e1cp-3},
    {0x1.d281c49d818d0p-1, 0x1.e199061890341p-3},
    {0x1.d4970f9ce00d9p-1, 0x1.cfb6b7b59d4dep-3},
    {0x1.d6986cfa798e7p-1, 0x1.be46a0a6082cbp-3},
    {0x1.d8865d98abe01p-1, 0x1.ad48bc25771c7p-3},
    {0x1.da61623cb41e0p-1, 0x1.9cbcdb9e90aaep-3},
    {0x1.dc29fb60715afp-1, 0x1.8ca2a85957ec6p-3},
    {0x1.dde0a90611a0dp-1, 0x1.7cf9a531a403fp-3},
    {0x1.df85ea8db188ep-1, 0x1.6dc1305420a79p-3},
    {0x1.e11a3e8cf4eb8p-1, 0x1.5ef885004f59cp-3},
    {0x1.e29e22a89d766p-1, 0x1.509ebd4e0c2a8p-3},
    {0x1.e4121370224ccp-1, 0x1.42b2d3f524f34p-3},
    {0x1.e5768c3b4a3fcp-1, 0x1.3533a6159f0c4p-3},
    {0x1.e6cc0709c8a0dp-1, 0x1.281ff4ff555ebp-3},
    {0x1.e812fc64db369p-1, 0x1.1b7667f7a7550p-3},
    {0x1.e94be342e6743p-1, 0x1.0f358dfc00722p-3},
    {0x1.ea7730ed0bbb9p-1, 0x1.035bdf80102bbp-3},
    {0x1.eb9558e6b42cep-1, 0x1.efcf804d33da1p-4},
    {0x1.eca6ccd709544p-1, 0x1.d9af00e7aba73p-4},
    {0x1.edabfc7453e63p-1, 0x1.c452bef0d750cp-4},
    {0x1.eea5557137ae0p-1, 0x1.afb718e8457f7p-4},
    {0x1.ef93436bc2daap-1, 0x1.9bd850dee55d4p-4},
    {0x1.f0762fde45ee6p-1, 0x1.88b28f966424fp-4},
    {0x1.f14e8211e8c55p-1, 0x1.7641e78b63dc8p-4},
    {0x1.f21c9f12f0677p-1, 0x1.648257e94a907p-4},
    {0x1.f2e0e9a6a8b09p-1, 0x1.536fcf668b5ebp-4},
    {0x1.f39bc242e43e6p-1, 0x1.43062f086c19ep-4},
    {0x1.f44d870704911p-1, 0x1.33414ccd6b2c7p-4},
    {0x1.f4f693b67bd77p-1, 0x1.241cf63d898b0p-4},
    {0x1.f59741b4b97cfp-1, 0x1.1594f2dfdbda5p-4},
    {0x1.f62fe80272419p-1, 0x1.07a50694e4566p-4},
    {0x1.f6c0db3c34641p-1, 0x1.f491e7aaa8e42p-5},
    {0x1.f74a6d9a38383p-1, 0x1.daf8fba9e2f70p-5},
    {0x1.f7cceef15d631p-1, 0x1.c276d512e5819p-5},
    {0x1.f848acb544e95p-1, 0x1.ab03092a9353ep-5},
    {0x1.f8bdf1fb78370p-1, 0x1.94953a2cb9ee0p-5},
    {0x1.f92d077f8d56dp-1, 0x1.7f251ab1af77bp-5},
    {0x1.f99633a838a57p-1, 0x1.6aaa70dc8596dp-5},
    {0x1.f9f9ba8d3c733p-1, 0x1.571d195267fdbp-5},
    {0x1.fa57ddfe27376p-1, 0x1.447509fbe441bp-5},
    {0x1.fab0dd89d1309p-1, 0x1.32aa5490fc7cap-5},
    {0x1.fb04f6868a944p-1, 0x1.21b528f107646p-5},
    {0x1.fb54641aebbc9p-1, 0x1.118dd7477eebcp-5},
    {0x1.fb9f5f4739170p-1, 0x1.022cd1fefa23cp-5},
    {0x1.fbe61eef4cf6ap-1, 0x1.e7155f0750059p-6},
    {0x1.fc28d7e4f9cd0p-1, 0x1.cb4057ad6df05p-6},
    {0x1.fc67bcf2d7b8fp-1, 0x1.b0cc53e851ab0p-6},
    {0x1.fca2fee770c79p-1, 0x1.97ab6a194752fp-6},
    {0x1.fcdacca0bfb73p-1, 0x1.7fd00329bd7e8p-6},
    {0x1.fd0f5317f582fp-1, 0x1.692cdc58ae482p-6},
    {0x1.fd40bd6d7a785p-1, 0x1.53b508ba01e10p-6},
    {0x1.fd6f34f52013ap-1, 0x1.3f5bf26b6469bp-6},
    {0x1.fd9ae142795e3p-1, 0x1.2c155b8213cf4p-6},
    {0x1.fdc3e835500b3p-1, 0x1.19d55eb5315c0p-6},
    {0x1.fdea6e062d0c9p-1, 0x1.08906fc825c07p-6},
    {0x1.fe0e9552ebdd6p-1, 0x1.f076b7714ba1ep-7},
    {0x1.fe307f2b503d0p-1, 0x1.d1969167c47a6p-7},
    {0x1.fe504b1d9696cp-1, 0x1.b46b6baccac7cp-7},
    {0x1.fe6e1742f7cf6p-1, 0x1.98e0f57430911p-7},
    {0x1.fe8a004c19ae6p-1, 0x1.7ee38dabb5b38p-7},
    {0x1.fea4218d6594ap-1, 0x1.6660416418b23p-7},
    {0x1.febc950b3fa75p-1, 0x1.4f44c9ea9e213p-7},
    {0x1.fed37386190fbp-1, 0x1.397f8a997d8cdp-7},
    {0x1.fee8d486585eep-1, 0x1.24ff8e657798bp-7},
    {0x1.fefcce6813974p-1, 0x1.11b4852eaa984p-7},
    {0x1.ff0f766697c76p-1, 0x1.ff1d81b5131bbp-8},
    {0x1.ff20e0a7ba8c2p-1, 0x1.dcfe64794b483p-8},
    {0x1.ff312046f2339p-1, 0x1.bceecba7888ddp-8},
    {0x1.ff404760319b4p-1, 0x1.9ed300c108a17p-8},
    {0x1.ff4e671a85425p-1, 0x1.829076b5375e1p-8},
    {0x1.ff5b8fb26f5f6p-1, 0x1.680dc292f9812p-8},
    {0x1.ff67d08401202p-1, 0x1.4f329409efa48p-8},
    {0x1.ff733814af88cp-1, 0x1.37e7adc463a6dp-8},
    {0x1.ff7dd41ce2b4dp-1, 0x1.2216dda21bc77p-8},
    {0x1.ff87b1913e853p-1, 0x1.0daaf4dbd8082p-8},
    {0x1.ff90dcaba4096p-1, 0x1.f51f802d90c77p-9},
    {0x1.ff9960f3eb327p-1, 0x1.d163feddab22dp-9},
    {0x1.ffa14948549a7p-1, 0x1.affebcfc45847p-9},
    {0x1.ffa89fe5b3625p-1, 0x1.90ccd8cf7ade9p-9},
    {0x1.ffaf6e6f4f5c0p-1, 0x1.73ad27d602858p-9},
    {0x1.ffb5bdf67fe6fp-1, 0x1.5880270993620p-9},
    {0x1.ffbb970200110p-1, 0x1.3f27eb464280ap-9},
    {0x1.ffc10194fcb64p-1, 0x1.278811df7007ep-9},
    {0x1.ffc60535dd7f5p-1, 0x1.1185b16a0f4b5p-9},
    {0x1.ffcaa8f4c9beap-1, 0x1.fa0e9586aebc7p-10},
    {0x1.ffcef371ea4d7p-1, 0x1.d3e974b462f89p-10},
    {0x1.ffd2eae369a07p-1, 0x1.b06e538214368p-10},
    {0x1.ffd6951b33686p-1, 0x1.8f72031a0154cp-10},
    {0x1.ffd9f78c7524ap-1, 0x1.70cbb70da2228p-10},
    {0x1.ffdd1750e1220p-1, 0x1.5454ea6271fbcp-10},
    {0x1.ffdff92db56e5p-1, 0x1.39e945501416ep-10},
    {0x1.ffe2a1988857cp-1, 0x1.216683b52187dp-10},
    {0x1.ffe514bbdc197p-1, 0x1.0aac5c46eedb6p-10},
    {0x1.ffe7567b7b5e1p-1, 0x1.eb38d0ff499f9p-11},
    {0x1.ffe96a78a04a9p-1, 0x1.c4341a9a49d9bp-11},
    {0x1.ffeb5415e7c44p-1, 0x1.a014c904be97ep-11},
    {0x1.ffed167b12ac2p-1, 0x1.7ea84e17f4e93p-11},
    {0x1.ffeeb49896c6dp-1, 0x1.5fbf2fd0f0e55p-11},
    {0x1.fff0312b010b5p-1, 0x1.432cdfc6b99abp-11},
    {0x1.fff18ebe2b0e1p-1, 0x1.28c794247ac65p-11},
    {0x1.fff2cfb0453d9p-1, 0x1.1068222437d65p-11},
    {0x1.fff3f634b79f9p-1, 0x1.f3d3b40b99f00p-12},
    {0x1.fff50456dab8cp-1, 0x1.ca54c8fa29f77p-12},
    {0x1.fff5fbfc8a439p-1, 0x1.a4134322792dep-12},
    {0x1.fff6dee89352ep-1, 0x1.80d311cd27e54p-12},
    {0x1.fff7aebcff755p-1, 0x1.605c16d71ad10p-12},
    {0x1.fff86cfd3e657p-1, 0x1.4279ecc2156f6p-12},
    {0x1.fff91b102fca8p-1, 0x1.26fbaf6b3f76fp-12},
    {0x1.fff9ba420e834p-1, 0x1.0db3c75613576p-12},
    {0x1.fffa4bc63ee9ap-1, 0x1.ecef6ef30c4a0p-13},
    {0x1.fffad0b901755p-1, 0x1.c23fdaf957587p-13},
    {0x1.fffb4a210b172p-1, 0x1.9b0f289f5395bp-13},
    {0x1.fffbb8f1049c6p-1, 0x1.7718d21af4ea3p-13},
    {0x1.fffc1e08f25f5p-1, 0x1.561d242583d44p-13},
    {0x1.fffc7a37857d2p-1, 0x1.37e0f06bb92fdp-13},
    {0x1.fffcce3b57bffp-1, 0x1.1c2d4418782dfp-13},
    {0x1.fffd1ac4135f9p-1, 0x1.02cf22526545ap-13},
    {0x1.fffd607387b07p-1, 0x1.d72e85099ad1dp-14},
    {0x1.fffd9fdeabccep-1, 0x1.acb3a4994cd3fp-14},
    {0x1.fffdd98e903b2p-1, 0x1.85dc75c5c9d7ap-14},
    {0x1.fffe0e0140857p-1, 0x1.625dd3bbe4b61p-14},
    {0x1.fffe3daa95b18p-1, 0x1.41f23a4966763p-14},
    {0x1.fffe68f4fa777p-1, 0x1.245963dc918c7p-14},
    {0x1.fffe904222101p-1, 0x1.0957ed550b883p-14},
    {0x1.fffeb3ebb267bp-1, 0x1.e16dfebfac43bp-15},
    {0x1.fffed443e2787p-1, 0x1.b487fa33a8f26p-15},
    {0x1.fffef1960d85dp-1, 0x1.8ba06f6c86e7ap-15},
    {0x1.ffff0c273bea2p-1, 0x1.66614dd110e9ap-15},
    {0x1.ffff2436a21dcp-1, 0x1.447b4ba5889f3p-15},
    {0x1.ffff39fe16963p-1, 0x1.25a568795ba85p-15},
    {0x1.ffff4db27f146p-1, 0x1.099c77b0a8d21p-15},
    {0x1.ffff5f8435efcp-1, 0x1.e045657233679p-16},
    {0x1.ffff6f9f67e55p-1, 0x1.b1fea4fbb871ap-16},
    {0x1.ffff7e2c6aea2p-1, 0x1.87fc5f659b544p-16},
    {0x1.ffff8b500e77cp-1, 0x1.61ded3265285bp-16},
    {0x1.ffff972be5c59p-1, 0x1.3f4e2568866c7p-16},
    {0x1.ffffa1de8c582p-1, 0x1.1ff9c722056c9p-16},
    {0x1.ffffab83e54b8p-1, 0x1.0397e4edcdab4p-16},
    {0x1.ffffb43555b5fp-1, 0x1.d3c9c205a0ffap-17},
    {0x1.ffffbc09fa7cdp-1, 0x1.a545ad51e9368p-17},
    {0x1.ffffc316d9ed0p-1, 0x1.7b324d2b1b3fap-17},
    {0x1.ffffc96f1165ep-1, 0x1.5528173ffd469p-17},
    {0x1.ffffcf23ff5fcp-1, 0x1.32c86e8d0bd8ap-17},
    {0x1.ffffd4456a10dp-1, 0x1.13bceb04817b8p-17},
    {0x1.ffffd8e1a2f22p-1, 0x1.ef6d5dc130f34p-18},
    {0x1.ffffdd05a75eap-1, 0x1.bcdb91720c06dp-18},
    {0x1.ffffe0bd3e852p-1, 0x1.8f414302d27abp-18},
    {0x1.ffffe41314e06p-1, 0x1.6626eb4552dfap-18},
    {0x1.ffffe710d565ep-1, 0x1.411fb0da07713p-18},
    {0x1.ffffe9bf4098cp-1, 0x1.1fc88257a4b03p-18},
    {0x1.ffffec2641a9ep-1, 0x1.01c7425dcd2f4p-18},
    {0x1.ffffee4d01cd6p-1, 0x1.cd94089e8db04p-19},
    {0x1.fffff039f9e8fp-1, 0x1.9d0cb1078fb5bp-19},
    {0x1.fffff1f302bc1p-1, 0x1.71714da87dc9cp-19},
    {0x1.fffff37d63a36p-1, 0x1.4a472cecbf851p-19},
    {0x1.fffff4dde0118p-1, 0x1.271f045a80a93p-19},
    {0x1.fffff618c3da6p-1, 0x1.0793efc9eef8dp-19},
    {0x1.fffff731ee681p-1, 0x1.d6950b79f9984p-20},
    {0x1.fffff82cdcf1bp-1, 0x1.a3dffe7e4b6e7p-20},
    {0x1.fffff90cb3c81p-1, 0x1.7672e3a0372c6p-20},
    {0x1.fffff9d446cccp-1, 0x1.4dc633ec4b4bfp-20},
    {0x1.fffffa8621251p-1, 0x1.295f6a5ace67bp-20},
    {0x1.fffffb248c39dp-1, 0x1.08cfd4008c875p-20},
    {0x1.fffffbb196132p-1, 0x1.d766f4ab4b806p-21},
    {0x1.fffffc2f171e3p-1, 0x1.a3604afdb0929p-21},
    {0x1.fffffc9eb76acp-1, 0x1.74e8e957fbd3ep-21},
    {0x1.fffffd01f36afp-1, 0x1.4b6e1584a8971p-21},
    {0x1.fffffd5a2041fp-1, 0x1.266b9b558b257p-21},
    {0x1.fffffda86faa9p-1, 0x1.056a6d77bd67cp-21},
    {0x1.fffffdedf37edp-1, 0x1.cffecb523a6b5p-22},
    {0x1.fffffe2ba0ea5p-1, 0x1.9b9443611cf54p-22},
    {0x1.fffffe62534d4p-1, 0x1.6ce7f55b086d3p-22},
    {0x1.fffffe92ced93p-1, 0x1.435e2906576d2p-22},
    {0x1.fffffebdc2ec6p-1, 0x1.1e6b06a04c886p-22},
    {0x1.fffffee3cc32cp-1, 0x1.fb221434d9775p-23},
    {0x1.ffffff0576917p-1, 0x1.c0bf364f50045p-23},
    {0x1.ffffff233ee1dp-1, 0x1.8ce38dc5ae5ddp-23},
    {0x1.ffffff3d9480fp-1, 0x1.5eda30351b6eep-23},
    {0x1.ffffff54dab72p-1, 0x1.36011717bbc77p-23},
    {0x1.ffffff6969fb8p-1, 0x1.11c73b1d86255p-23},
    {0x1.ffffff7b91176p-1, 0x1.e355bbaee85cbp-24},
    {0x1.ffffff8b962bep-1, 0x1.aa6ffb0ba51a0p-24},
    {0x1.ffffff99b79d2p-1, 0x1.780dde696d57cp-24},
    {0x1.ffffffa62ce54p-1, 0x1.4b763749e3996p-24},
    {0x1.ffffffb127525p-1, 0x1.2403b79962533p-24},
    {0x1.ffffffbad2affp-1, 0x1.0122e403955bbp-24},
    {0x1.ffffffc355dfdp-1, 0x1.c4a07483a366dp-25},
    {0x1.ffffffcad3626p-1, 0x1.8e2d0d030ee58p-25},
    {0x1.ffffffd169d0cp-1, 0x1.5e1ac6dedefcap-25},
    {0x1.ffffffd7344aap-1, 0x1.33afc1b2bdc4fp-25},
    {0x1.ffffffdc4ad7ap-1, 0x1.0e469a6b398d7p-25},
    {0x1.ffffffe0c2bf0p-1, 0x1.da987acf4f2d9p-26},
    {0x1.ffffffe4aed5ep-1, 0x1.a07be3274183bp-26},
    {0x1.ffffffe81fc4ep-1, 0x1.6d4f2dd6f71b4p-26},
    {0x1.ffffffeb24467p-1, 0x1.404426c3f1810p-26},
    {0x1.ffffffedc95e7p-1, 0x1.18a3d329db37cp-26},
    {0x1.fffffff01a8b6p-1, 0x1.eb97d4afc3bd3p-27},
    {0x1.fffffff221f30p-1, 0x1.ae59247f070adp-27},
    {0x1.fffffff3e8892p-1, 0x1.788cb21027cf8p-27},
    {0x1.fffffff57632dp-1, 0x1.4950caffea471p-27},
    {0x1.fffffff6d1e56p-1, 0x1.1fddb1b6cdf3dp-27},
    {0x1.fffffff801c1fp-1, 0x1.f70572e880ffep-28},
    {0x1.fffffff90b2e3p-1, 0x1.b74763a7056c0p-28},
    {0x1.fffffff9f2e9fp-1, 0x1.7f6d3332815fdp-28},
    {0x1.fffffffabd229p-1, 0x1.4e8322cdbc100p-28},
    {0x1.fffffffb6d844p-1, 0x1.23b20f56b83b6p-28},
    {0x1.fffffffc0748fp-1, 0x1.fc785f4cc55d5p-29},
    {0x1.fffffffc8d462p-1, 0x1.baf45d47a63b0p-29},
    {0x1.fffffffd01f89p-1, 0x1.81b12ead7e725p-29},
    {0x1.fffffffd678edp-1, 0x1.4fab14805e6a5p-29},
    {0x1.fffffffdbff2ap-1, 0x1.23fd68479eb54p-29},
    {0x1.fffffffe0cd16p-1, 0x1.fbbdfce63ed31p-30},
    {0x1.fffffffe4fa30p-1, 0x1.b93de1e27ca3bp-30},
    {0x1.fffffffe89b0cp-1, 0x1.7f438d5016e96p-30},
    {0x1.fffffffebc1a9p-1, 0x1.4cbddb5f789e9p-30},
    {0x1.fffffffee7dc8p-1, 0x1.20bcfe77e3b39p-30},
    {0x1.ffffffff0dd2bp-1, 0x1.f4dd14577e044p-31},
    {0x1.ffffffff2ebdap-1, 0x1.b233e5953c928p-31},
    {0x1.ffffffff4b453p-1, 0x1.783ae930d011ep-31},
    {0x1.ffffffff63fc3p-1, 0x1.45d6ae286fa0ep-31},
    {0x1.ffffffff79626p-1, 0x1.1a0f03f106cd8p-31},
    {0x1.ffffffff8be77p-1, 0x1.e8156af08d0d8p-32},
    {0x1.ffffffff9bec8p-1, 0x1.a617897179d8ap-32},
    {0x1.ffffffffa9c63p-1, 0x1.6cd830779f7cbp-32},
    {0x1.ffffffffb5be5p-1, 0x1.3b351b01e9334p-32},
    {0x1.ffffffffc014ep-1, 0x1.1030c9635f40ep-32},
    {0x1.ffffffffc901cp-1, 0x1.d5dbed4c4fe10p-33},
    {0x1.ffffffffd0b56p-1, 0x1.9557332ea02aep-33},
    {0x1.ffffffffd759dp-1, 0x1.5d82c26ce1c09p-33},
    {0x1.ffffffffdd13cp-1, 0x1.2d393c321d0b2p-33},
    {0x1.ffffffffe202dp-1, 0x1.037b17e7291e0p-33},
    {0x1.ffffffffe642ap-1, 0x1.bed3bfb983a47p-34},
    {0x1.ffffffffe9eb0p-1, 0x1.808806e465fddp-34},
    {0x1.ffffffffed10ap-1, 0x1.4ac259d756915p-34},
    {0x1.ffffffffefc57p-1, 0x1.1c5e1671310bbp-34},
    {0x1.fffffffff218fp-1, 0x1.e8ba06f579b7fp-35},
    {0x1.fffffffff4188p-1, 0x1.a3c4c749fa106p-35},
    {0x1.fffffffff5cfdp-1, 0x1.685d4c6df2e9fp-35},
    {0x1.fffffffff748ep-1, 0x1.35374479d0248p-35},
    {0x1.fffffffff88c5p-1, 0x1.0932969ba7c57p-35},
    {0x1.fffffffff9a1bp-1, 0x1.c6ab43f84aea0p-36},
    {0x1.fffffffffa8f6p-1, 0x1.85906f6d14650p-36},
    {0x1.fffffffffb5b0p-1, 0x1.4d9e7182dff92p-36},
    {0x1.fffffffffc095p-1, 0x1.1d9186da6a5abp-36},
    {0x1.fffffffffc9e8p-1, 0x1.e8a37a45fc32ep-37},
    {0x1.fffffffffd1e1p-1, 0x1.a1da4ab9a1531p-37},
    {0x1.fffffffffd8b3p-1, 0x1.65258cbfca61fp-37},
    {0x1.fffffffffde86p-1, 0x1.311c6eca3f484p-37},
    {0x1.fffffffffe380p-1, 0x1.04879a92986b8p-37},
    {0x1.fffffffffe7c0p-1, 0x1.bcb51f852a3b3p-38},
    {0x1.fffffffffeb60p-1, 0x1.7b5bbc16d67abp-38},
    {0x1.fffffffffee77p-1, 0x1.4374441235915p-38},
    {0x1.ffffffffff11ap-1, 0x1.13a757c355f22p-38},
    {0x1.ffffffffff359p-1, 0x1.d59ae6d0dc693p-39},
    {0x1.ffffffffff542p-1, 0x1.8fd0cab75acbfp-39},
    {0x1.ffffffffff6e3p-1, 0x1.543b4818f8935p-39},
    {0x1.ffffffffff845p-1, 0x1.2162cd16ab8aep-39},
    {0x1.ffffffffff973p-1, 0x1.ec099892b29ccp-40},
    {0x1.ffffffffffa73p-1, 0x1.a218cb2a40dd0p-40},
    {0x1.ffffffffffb4cp-1, 0x1.63181ba056531p-40},
    {0x1.ffffffffffc05p-1, 0x1.2d7026e60ab5ep-40},
    {0x1.ffffffffffca2p-1, 0x1.ff878b9f1e143p-41},
    {0x1.ffffffffffd27p-1, 0x1.b1cfc37ee5895p-41},
    {0x1.ffffffffffd98p-1, 0x1.6fb8d1b65e748p-41},
    {0x1.ffffffffffdf8p-1, 0x1.378c76327f5a3p-41},
    {0x1.ffffffffffe49p-1, 0x1.07d3dd1d4acd5p-41},
    {0x1.ffffffffffe8dp-1, 0x1.be9d37424eee7p-42},
    {0x1.ffffffffffec7p-1, 0x1.79d5dc6f8d9f9p-42},
    {0x1.ffffffffffef8p-1, 0x1.3f7e194466984p-42},
    {0x1.fffffffffff22p-1, 0x1.0e06db0545094p-42},
    {0x1.fffffffffff45p-1, 0x1.c83762a20dfaep-43},
    {0x1.fffffffffff62p-1, 0x1.8134ae32bfcb3p-43},
    {0x1.fffffffffff7bp-1, 0x1.4516dd5166117p-43},
    {0x1.fffffffffff90p-1, 0x1.12388c210f82fp-43},
    {0x1.fffffffffffa2p-1, 0x1.ce65fc9e07b69p-44},
    {0x1.fffffffffffb1p-1, 0x1.85a9ed123f0f2p-44},
    {0x1.fffffffffffbep-1, 0x1.4835bd010a41bp-44},
    {0x1.fffffffffffc8p-1, 0x1.1450202d4e4e1p-44},
    {0x1.fffffffffffd1p-1, 0x1.d1045b6d112d0p-45},
    {0x1.fffffffffffd9p-1, 0x1.871b1aa423baep-45},
    {0x1.fffffffffffdfp-1, 0x1.48c824472e49ap-45},
    {0x1.fffffffffffe4p-1, 0x1.14411e12964d5p-45},
    {0x1.fffffffffffe9p-1, 0x1.d002ddf03ef28p-46},
    {0x1.fffffffffffedp-1, 0x1.857f99bfe8fbbp-46},
    {0x1.ffffffffffff0p-1, 0x1.46caa8412b080p-46},
    {0x1.ffffffffffff3p-1, 0x1.120bdf83abdafp-46},
    {0x1.ffffffffffff5p-1, 0x1.cb6786c50ff4fp-47},
    {0x1.ffffffffffff7p-1, 0x1.80e104066ffacp-47},
    {0x1.ffffffffffff8p-1, 0x1.42492928e267cp-47},
    {0x1.ffffffffffff9p-1, 0x1.0dbd8d82578a6p-47},
    {0x1.ffffffffffffbp-1, 0x1.c34dc092042e6p-48},
    {0x1.ffffffffffffbp-1, 0x1.795aca9287d3bp-48},
    {0x1.ffffffffffffcp-1, 0x1.3b5e5c86b9440p-48},
    {0x1.ffffffffffffdp-1, 0x1.076f9dfb1c661p-48},
    {0x1.ffffffffffffdp-1, 0x1.b7e54ec9b3dabp-49},
    {0x1.ffffffffffffep-1, 0x1.6f1926fb4b8f0p-49},
    {0x1.ffffffffffffep-1, 0x1.3232c60248eb0p-49},
    {0x1.ffffffffffffep-1, 0x1.fe8db307aa9b7p-50},
    {0x1.fffffffffffffp-1, 0x1.a970798776731p-50},
    {0x1.fffffffffffffp-1, 0x1.62576b411f78cp-50},
    {0x1.fffffffffffffp-1, 0x1.26fb2cf70e351p-50},
    {0x1.fffffffffffffp-1, 0x1.eae3ed4fe32d1p-51},
    {0x1.fffffffffffffp-1, 0x1.98418d8c5509fp-51},
    {0x1.0000000000000p+0, 0x1.535dc7ab7081ap-51},
    {0x1.0000000000000p+0, 0x1.19f6a3be40417p-51},
    {0x1.0000000000000p+0, 0x1.d44fbb3f2f179p-52},
    {0x1.0000000000000p+0, 0x1.84b7d20f7ce81p-52},
    {0x1.0000000000000p+0, 0x1.427ea477f2f18p-52},
    {0x1.0000000000000p+0, 0x1.0b6c3afdde064p-52},
};

// a constant the compiler keeps in scalar registers: as plain literals the
// coefficients below are hoisted out of the callers' loops into some 40
// vector registers
__device__ __forceinline__ double scalar(double v) {
    long long b = __builtin_bit_cast(long long, v);
    asm("" : "+s"(b));
    return __builtin_bit_cast(double, b);
}

// exp(x) by its Taylor series to x^13 on |r| <= ln(2)/2, x = n*ln(2) + r with
// ln(2) in two parts (n times the first is exact for |n| < 2^12): 0.8 ulp.
// Results beyond the range of doubles are 0 and infinity, infinite x included:
// below -1500, where exp is 0, -1500 takes x's place, since r, and with it the
// polynomial's sign, would follow x down (a NaN compares false and stays); far
// above, r and the polynomial grow with x and the result is infinity anyway.
__device__ __forceinline__ double exp_series(double x) {
    x = x < -1500.0 ? -1500.0 : x;
    const double n = __builtin_fmin(__builtin_rint(x * scalar(1.4426950408889634)), 2100.0);
    double r = fma(n, scalar(-0x1.62e42fefap-1), x);
    r = fma(n, scalar(-0x1.cf79abc9e3b3ap-40), r);
    double a = scalar(1.0 / 6227020800.0);
    a = fma(r, a, scalar(1.0 / 479001600.0));
    a = fma(r, a, scalar(1.0 / 39916800.0));
    a = fma(r, a, scalar(1.0 / 3628800.0));
    a = fma(r, a, scalar(1.0 / 362880.0));
    a = fma(r, a, scalar(1.0 / 40320.0));
    a = fma(r, a, scalar(1.0 / 5040.0));
    a = fma(r, a, scalar(1.0 / 720.0));
    a = fma(r, a, scalar(1.0 / 120.0));
    a = fma(r, a, scalar(1.0 / 24.0));
    a = fma(r, a, scalar(1.0 / 6.0));
    a = fma(r, a, 0.5);
    a = fma(r, a, 1.0);
    a = fma(r, a, 1.0);
    return __builtin_ldexp(a, (int)n);
}

// the workgroup's copy of the table: random reads of 16 bytes cost LDS little,
// where through the vector cache they would compete with the gathers
__device__ __forceinline__ double2* erf_nodes() {
    __shared__ double2 nodes[kErfNodes];
    return nodes;
}

// every thread of a workgroup, before the first erf_exp
__device__ __forceinline__ void load_erf_nodes() {
    double2* n = erf_nodes();
    for (int j = (int)threadIdx.x; j < kErfNodes; j += (int)blockDim.x)
        n[j] = make_double2(kErfTable[j][0], kErfTable[j][1]);
    __syncthreads();
}

__device__ __forceinline__ void erf_exp(double x, double& er, double& ex) {
    const double ax = __builtin_fabs(x);
    const double jf = __builtin_rint(ax * 64.0);
    // beyond the table (infinity included) and for NaN any node will do
    const int j = (int)__builtin_fmin(jf, kErfNodes - 1.0);
    const double2 node = erf_nodes()[j];
    const double d = fma(jf, -0.015625, ax);
    const double p = (jf * -0.03125) * d, s = d * d;
    double a0 = fma(p, scalar(1.0 / 362880.0), scalar(1.0 / 40320.0));
    a0 = fma(p, a0, scalar(1.0 / 5040.0));
    a0 = fma(p, a0, scalar(1.0 / 720.0));
    a0 = fma(p, a0, scalar(1.0 / 120.0));
    a0 = fma(p, a0, scalar(1.0 / 24.0));
    a0 = fma(p, a0, scalar(1.0 / 6.0));
    a0 = fma(p, a0, 0.5);
    a0 = fma(p, a0, 1.0);
    double a1 = fma(p, scalar(1.0 / 168.0), scalar(1.0 / 36.0));
    a1 = fma(p, a1, scalar(0.1));
    a1 = fma(p, a1, scalar(0.25));
    a1 = fma(p, a1, scalar(1.0 / 3.0));
    double a2 = fma(p, scalar(1.0 / 28.0), scalar(1.0 / 12.0));
    a2 = fma(p, a2, scalar(0.1));
    double t = fma(s, scalar(-1.0 / 42.0), a2);
    t = fma(s, t, -a1);
    const double u = d * fma(s, t, a0);
    const double a = p * a0;
    const double b = s * fma(s, fma(s, scalar(-1.0 / 6.0), 0.5), -1.0);
    ex = fma(node.y, fma(a, b, a) + b, node.y);
    double e = fma(scalar(1.1283791670955126) * node.y, u, node.x);
    if (ax > 6.0) {
        e = 1.0;
        ex = exp_series(-x * x);
    }
    er = __builtin_copysign(e, x);
}

}  // namespace mfcfd
