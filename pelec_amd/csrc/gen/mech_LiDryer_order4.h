// GENERATED by pelec_amd/mechgen.py -- do not edit.
// mechanism: LiDryer_order4  source sha256: de6aa08e8a9f786b4e05399c596fafa946a36809c9fa4429ec7903cd7502ba7f
// species: 9  reactions: 22
#pragma once
#include <cmath>
#include <cstdint>
#ifndef PELEC_MEMORY_FENCE
#define PELEC_MEMORY_FENCE() __asm__ __volatile__("" ::: "memory")
#endif
#ifndef PELEC_REG_CHAIN
#if defined(__HIP_DEVICE_COMPILE__)
#define PELEC_REG_CHAIN(a, b, c, d) __asm__ __volatile__("" : "+v"(a), "+v"(b), "+v"(c) : "v"(d))
#else
#define PELEC_REG_CHAIN(a, b, c, d) ((void)(d))
#endif
#endif
// RMUL(k, j): the rate constant of reaction j times its multiplier rmul[j] when MUL (the
// per-reaction pre-exponential scaling exp(log A_j) of the sensitivity and adjoint paths)
#ifndef RMUL
#define RMUL_DEF (void)rmul
#define RMUL(k, j) (MUL ? (k) * rmul[j] : (k))
#endif
#ifndef __HIPCC__
#define __host__
#define __device__
#endif
namespace pelec {
namespace mech {
struct LiDryer_order4 {
  static constexpr int NSP = 9;
  static constexpr int NRXN = 22;
  static constexpr const char* NAME = "LiDryer_order4";
  static constexpr const char* SHA256 = "de6aa08e8a9f786b4e05399c596fafa946a36809c9fa4429ec7903cd7502ba7f";
  static constexpr double W[9] = {2.01594, 31.9988, 18.01534, 1.00797, 15.9994, 17.007369999999998, 33.006769999999996, 34.014739999999996, 28.0134};
  static constexpr double IW[9] = {0.49604650932071387, 0.03125117191894696, 0.055508250191225926, 0.9920930186414277, 0.06250234383789392, 0.05879803873262004, 0.03029681486555637, 0.02939901936631002, 0.03569720205330306};
  static constexpr const char* SPECIES[9] = {"H2", "O2", "H2O", "H", "O", "OH", "HO2", "H2O2", "N2"};
  // ---- thermo: folded NASA-7 polynomials (mass units, erg/g, erg/(g K))
  __host__ __device__ static inline void tmid_flags(double T, bool* lo) {
    lo[0] = T < 1000.0;
  }
  // species e_k, cv_k (mass units) and dcv_k/dT
  __host__ __device__ static inline void e_cv(double T, double* e, double* cv) {
    bool lo[1]; tmid_flags(T, lo);
    e[0] = lo[0] ? fma(T, fma(T, fma(T, fma(T, fma(T, 3.4107402675524593e-06, -0.0009770025618790518), -11.194908878994598), 17011.834957792224), 94782910.65151145), -41760012721.584656) : fma(T, fma(T, fma(T, fma(T, fma(T, 1.3055678579528436e-08, -9.518588126080866e-05), -0.7745313289345194), 14436.58859911475), 82133456.80144538), -34439809606.868126);
    cv[0] = lo[0] ? fma(T, fma(T, fma(T, fma(T, 1.7053701337762297e-05, -0.003908010247516207), -33.584726636983795), 34023.66991558445), 94782910.65151145) : fma(T, fma(T, fma(T, fma(T, 6.527839289764218e-08, -0.00038074352504323465), -2.323593986803558), 28873.1771982295), 82133456.80144538);
    e[1] = lo[0] ? fma(T, fma(T, fma(T, fma(T, fma(T, -4.5567842824267206e-07, 0.0008534836619928971), -0.498553008232421), 1464.8112115909228), 5750019.890860144), -2612005835.355053) : fma(T, fma(T, fma(T, fma(T, fma(T, -5.905750419053826e-10, 1.153207894609931e-05), -0.1090311173248295), 797.0746732925282), 7009297.673835451), -3206203000.868104);
    cv[1] = lo[0] ? fma(T, fma(T, fma(T, fma(T, -2.2783921412133602e-06, 0.0034139346479715883), -1.495659024697263), 2929.6224231818455), 5750019.890860144) : fma(T, fma(T, fma(T, fma(T, -2.952875209526913e-09, 4.612831578439724e-05), -0.32709335197448847), 1594.1493465850565), 7009297.673835451);
    e[2] = lo[0] ? fma(T, fma(T, fma(T, fma(T, fma(T, -2.3136873603397435e-06, 0.00804037090419511), -9.776091253662699), 8018.89055042963), 11015783.540270746), -139416853281.73718) : fma(T, fma(T, fma(T, fma(T, fma(T, -5.899735328949149e-09, 0.00013857130016074593), -1.343066897743044), 7052.721152812942), 7717309.475754812), -137991214074.95697);
    cv[2] = lo[0] ? fma(T, fma(T, fma(T, fma(T, -1.1568436801698717e-05, 0.03216148361678044), -29.328273760988097), 16037.78110085926), 11015783.540270746) : fma(T, fma(T, fma(T, fma(T, -2.9498676644745744e-08, 0.0005542852006429837), -4.029200693229132), 14105.442305625884), 7717309.475754812);
    e[3] = lo[0] ? fma(T, fma(T, fma(T, fma(T, fma(T, 0.0, 0.0), 0.0), 0.0), 123730804.75837436), 2101083518938.3674) : fma(T, fma(T, fma(T, fma(T, fma(T, 0.0, 0.0), 0.0), 0.0), 123730804.75837436), 2101083518938.3674);
    cv[3] = lo[0] ? fma(T, fma(T, fma(T, fma(T, 0.0, 0.0), 0.0), 0.0), 123730804.75837436) : fma(T, fma(T, fma(T, fma(T, 0.0, 0.0), 0.0), 0.0), 123730804.75837436);
    e[4] = lo[0] ? fma(T, fma(T, fma(T, fma(T, fma(T, 4.043782448166599e-07, -0.0020823871842488772), 4.193819781023616), -4256.556486283742), 10115073.789885493), 151472532212.07553) : fma(T, fma(T, fma(T, fma(T, fma(T, -4.5399208805517084e-10, 5.912671169576799e-06), -0.005374813962813966), -71.58662202862139), 8013675.653430371), 151904692612.66907);
    cv[4] = lo[0] ? fma(T, fma(T, fma(T, fma(T, 2.0218912240832993e-06, -0.008329548736995509), 12.581459343070849), -8513.112972567484), 10115073.789885493) : fma(T, fma(T, fma(T, fma(T, -2.269960440275854e-09, 2.3650684678307196e-05), -0.016124441888441896), -143.17324405724278), 8013675.653430371);
    e[5] = lo[0] ? fma(T, fma(T, fma(T, fma(T, fma(T, 2.0164822405361935e-06, -0.0070868856247666085), 10.637324920058875), -7884.193258540319), 15278809.51884366), 16359238477.301249) : fma(T, fma(T, fma(T, fma(T, fma(T, -1.302320266912726e-09, 3.7303375762027e-05), -0.42219616287900336), 2582.488357950532), 9116176.33970538), 18008306717.04652);
    cv[5] = lo[0] ? fma(T, fma(T, fma(T, fma(T, 1.0082411202680968e-05, -0.028347542499066434), 31.911974760176626), -15768.386517080638), 15278809.51884366) : fma(T, fma(T, fma(T, fma(T, -6.51160133456363e-09, 0.000149213503048108), -1.26658848863701), 5164.976715901064), 9116176.33970538);
    e[6] = lo[0] ? fma(T, fma(T, fma(T, fma(T, fma(T, 4.681468412296513e-06, -0.015288161502173006), 17.766032421634424), -5981.558472625442), 8317286.461788826), 742626566.6440628) : fma(T, fma(T, fma(T, fma(T, fma(T, -5.436469429981671e-09, 7.194714695081523e-05), -0.5320652905311182), 2821.072880241255), 7600406.5951120015), 281769000.368105);
    cv[6] = lo[0] ? fma(T, fma(T, fma(T, fma(T, 2.3407342061482568e-05, -0.061152646008692024), 53.29809726490328), -11963.116945250884), 8317286.461788826) : fma(T, fma(T, fma(T, fma(T, -2.7182347149908354e-08, 0.0002877885878032609), -1.5961958715933544), 5642.14576048251), 7600406.5951120015);
    e[7] = lo[0] ? fma(T, fma(T, fma(T, fma(T, fma(T, 1.2082596590598668e-06, -0.0028267959027342975), -0.12099739775532213), 8028.811040037399), 5838999.75039175), -43175282361.06859) : fma(T, fma(T, fma(T, fma(T, fma(T, -6.998985536934612e-09, 0.0001435397896737607), -1.2015620839575023), 5299.561407676278), 8734143.91817158), -44015681374.1868);
    cv[7] = lo[0] ? fma(T, fma(T, fma(T, fma(T, 6.041298295299334e-06, -0.01130718361093719), -0.3629921932659664), 16057.622080074798), 5838999.75039175) : fma(T, fma(T, fma(T, fma(T, -3.499492768467306e-08, 0.0005741591586950428), -3.604686251872507), 10599.122815352555), 8734143.91817158);
    e[8] = lo[0] ? fma(T, fma(T, fma(T, fma(T, fma(T, -1.4512808516142303e-06, 0.004186047175392025), -3.9209879517709996), 2089.8496500582078), 6822543.492653029), -3030062358.3258877) : fma(T, fma(T, fma(T, fma(T, fma(T, -4.0088303766602985e-09, 7.492080721547366e-05), -0.5624181383151804), 2208.180574862709), 5718326.321916925), -2738891737.799691);
    cv[8] = lo[0] ? fma(T, fma(T, fma(T, fma(T, -7.256404258071151e-06, 0.0167441887015681), -11.762963855312998), 4179.6993001164155), 6822543.492653029) : fma(T, fma(T, fma(T, fma(T, -2.004415188330149e-08, 0.00029968322886189463), -1.6872544149455413), 4416.361149725418), 5718326.321916925);
  }
  __host__ __device__ static inline void dcv_dT(double T, double* d) {
    bool lo[1]; tmid_flags(T, lo);
    d[0] = lo[0] ? fma(T, fma(T, fma(T, 6.821480535104919e-05, -0.011724030742548621), -67.16945327396759), 34023.66991558445) : fma(T, fma(T, fma(T, 2.611135715905687e-07, -0.001142230575129704), -4.647187973607116), 28873.1771982295);
    d[1] = lo[0] ? fma(T, fma(T, fma(T, -9.113568564853441e-06, 0.010241803943914765), -2.991318049394526), 2929.6224231818455) : fma(T, fma(T, fma(T, -1.1811500838107651e-08, 0.0001383849473531917), -0.6541867039489769), 1594.1493465850565);
    d[2] = lo[0] ? fma(T, fma(T, fma(T, -4.627374720679487e-05, 0.09648445085034131), -58.656547521976194), 16037.78110085926) : fma(T, fma(T, fma(T, -1.1799470657898298e-07, 0.001662855601928951), -8.058401386458264), 14105.442305625884);
    d[3] = lo[0] ? fma(T, fma(T, fma(T, 0.0, 0.0), 0.0), 0.0) : fma(T, fma(T, fma(T, 0.0, 0.0), 0.0), 0.0);
    d[4] = lo[0] ? fma(T, fma(T, fma(T, 8.087564896333197e-06, -0.024988646210986527), 25.162918686141698), -8513.112972567484) : fma(T, fma(T, fma(T, -9.079841761103417e-09, 7.095205403492159e-05), -0.03224888377688379), -143.17324405724278);
    d[5] = lo[0] ? fma(T, fma(T, fma(T, 4.032964481072387e-05, -0.0850426274971993), 63.82394952035325), -15768.386517080638) : fma(T, fma(T, fma(T, -2.604640533825452e-08, 0.00044764050914432405), -2.53317697727402), 5164.976715901064);
    d[6] = lo[0] ? fma(T, fma(T, fma(T, 9.362936824593027e-05, -0.18345793802607607), 106.59619452980655), -11963.116945250884) : fma(T, fma(T, fma(T, -1.0872938859963342e-07, 0.0008633657634097827), -3.192391743186709), 5642.14576048251);
    d[7] = lo[0] ? fma(T, fma(T, fma(T, 2.4165193181197337e-05, -0.03392155083281157), -0.7259843865319328), 16057.622080074798) : fma(T, fma(T, fma(T, -1.3997971073869224e-07, 0.0017224774760851284), -7.209372503745014), 10599.122815352555);
    d[8] = lo[0] ? fma(T, fma(T, fma(T, -2.9025617032284605e-05, 0.05023256610470429), -23.525927710625997), 4179.6993001164155) : fma(T, fma(T, fma(T, -8.017660753320596e-08, 0.0008990496865856839), -3.3745088298910826), 4416.361149725418);
  }
  // mixture e(T) = sum Y_k e_k(T) as polynomial coefficients per Tmid group and range:
  // pe[(g*2 + b)*6 + i], g < 1 Tmid groups, b = 0 low / 1 high
  static constexpr int NTMID = 1;
  __host__ __device__ static inline void mix_e_poly(const double* Y, double* pe) {
    pe[0] = -41760012721.584656 * Y[0] + -2612005835.355053 * Y[1] + -139416853281.73718 * Y[2] + 2101083518938.3674 * Y[3] + 151472532212.07553 * Y[4] + 16359238477.301249 * Y[5] + 742626566.6440628 * Y[6] + -43175282361.06859 * Y[7] + -3030062358.3258877 * Y[8];
    pe[1] = 94782910.65151145 * Y[0] + 5750019.890860144 * Y[1] + 11015783.540270746 * Y[2] + 123730804.75837436 * Y[3] + 10115073.789885493 * Y[4] + 15278809.51884366 * Y[5] + 8317286.461788826 * Y[6] + 5838999.75039175 * Y[7] + 6822543.492653029 * Y[8];
    pe[2] = 17011.834957792224 * Y[0] + 1464.8112115909228 * Y[1] + 8018.89055042963 * Y[2] + -4256.556486283742 * Y[4] + -7884.193258540319 * Y[5] + -5981.558472625442 * Y[6] + 8028.811040037399 * Y[7] + 2089.8496500582078 * Y[8];
    pe[3] = -11.194908878994598 * Y[0] + -0.498553008232421 * Y[1] + -9.776091253662699 * Y[2] + 4.193819781023616 * Y[4] + 10.637324920058875 * Y[5] + 17.766032421634424 * Y[6] + -0.12099739775532213 * Y[7] + -3.9209879517709996 * Y[8];
    pe[4] = -0.0009770025618790518 * Y[0] + 0.0008534836619928971 * Y[1] + 0.00804037090419511 * Y[2] + -0.0020823871842488772 * Y[4] + -0.0070868856247666085 * Y[5] + -0.015288161502173006 * Y[6] + -0.0028267959027342975 * Y[7] + 0.004186047175392025 * Y[8];
    pe[5] = 3.4107402675524593e-06 * Y[0] + -4.5567842824267206e-07 * Y[1] + -2.3136873603397435e-06 * Y[2] + 4.043782448166599e-07 * Y[4] + 2.0164822405361935e-06 * Y[5] + 4.681468412296513e-06 * Y[6] + 1.2082596590598668e-06 * Y[7] + -1.4512808516142303e-06 * Y[8];
    pe[6] = -34439809606.868126 * Y[0] + -3206203000.868104 * Y[1] + -137991214074.95697 * Y[2] + 2101083518938.3674 * Y[3] + 151904692612.66907 * Y[4] + 18008306717.04652 * Y[5] + 281769000.368105 * Y[6] + -44015681374.1868 * Y[7] + -2738891737.799691 * Y[8];
    pe[7] = 82133456.80144538 * Y[0] + 7009297.673835451 * Y[1] + 7717309.475754812 * Y[2] + 123730804.75837436 * Y[3] + 8013675.653430371 * Y[4] + 9116176.33970538 * Y[5] + 7600406.5951120015 * Y[6] + 8734143.91817158 * Y[7] + 5718326.321916925 * Y[8];
    pe[8] = 14436.58859911475 * Y[0] + 797.0746732925282 * Y[1] + 7052.721152812942 * Y[2] + -71.58662202862139 * Y[4] + 2582.488357950532 * Y[5] + 2821.072880241255 * Y[6] + 5299.561407676278 * Y[7] + 2208.180574862709 * Y[8];
    pe[9] = -0.7745313289345194 * Y[0] + -0.1090311173248295 * Y[1] + -1.343066897743044 * Y[2] + -0.005374813962813966 * Y[4] + -0.42219616287900336 * Y[5] + -0.5320652905311182 * Y[6] + -1.2015620839575023 * Y[7] + -0.5624181383151804 * Y[8];
    pe[10] = -9.518588126080866e-05 * Y[0] + 1.153207894609931e-05 * Y[1] + 0.00013857130016074593 * Y[2] + 5.912671169576799e-06 * Y[4] + 3.7303375762027e-05 * Y[5] + 7.194714695081523e-05 * Y[6] + 0.0001435397896737607 * Y[7] + 7.492080721547366e-05 * Y[8];
    pe[11] = 1.3055678579528436e-08 * Y[0] + -5.905750419053826e-10 * Y[1] + -5.899735328949149e-09 * Y[2] + -4.5399208805517084e-10 * Y[4] + -1.302320266912726e-09 * Y[5] + -5.436469429981671e-09 * Y[6] + -6.998985536934612e-09 * Y[7] + -4.0088303766602985e-09 * Y[8];
  }
  __host__ __device__ static inline double tmid(int g) {
    if (g == 0) return 1000.0;
    return 0.0;
  }
  // g_k/RT and h_k/RT
  __host__ __device__ static inline void g_h_RT(double T, double lnT, double invT, double* gRT, double* hRT) {
    bool lo[1]; tmid_flags(T, lo);
    gRT[0] = lo[0] ? (fma(T, fma(T, fma(T, fma(T, -2.067436e-14, 7.896194999999999e-12), 1.3571691666666666e-07), -0.0004124721), 6.592218) - 3.298124 * lnT + -1012.521 * invT) : (fma(T, fma(T, fma(T, fma(T, -7.91376e-17, 7.692981666666667e-13), 9.389715e-09), -0.0003500322), 4.346533) - 2.991423 * lnT + -835.034 * invT);
    if (hRT) hRT[0] = lo[0] ? (fma(T, fma(T, fma(T, fma(T, 8.269744e-14, -2.3688585e-11), -2.714338333333333e-07), 0.0004124721), 3.298124) + -1012.521 * invT) : (fma(T, fma(T, fma(T, fma(T, 3.165504e-16, -2.3078945e-12), -1.877943e-08), 0.0003500322), 2.991423) + -835.034 * invT);
    gRT[1] = lo[0] ? (fma(T, fma(T, fma(T, fma(T, 4.384277e-14, -1.0948975000000001e-10), 9.593583333333333e-08), -0.000563743), -2.821802) - 3.212936 * lnT + -1005.249 * invT) : (fma(T, fma(T, fma(T, fma(T, 5.682175000000001e-17, -1.4794008333333333e-12), 2.09807e-08), -0.00030675985), 0.5084119999999999) - 3.697578 * lnT + -1233.93 * invT);
    if (hRT) hRT[1] = lo[0] ? (fma(T, fma(T, fma(T, fma(T, -1.7537108e-13, 3.2846925e-10), -1.9187166666666667e-07), 0.000563743), 3.212936) + -1005.249 * invT) : (fma(T, fma(T, fma(T, fma(T, -2.2728700000000004e-16, 4.4382025e-12), -4.19614e-08), 0.00030675985), 3.697578) + -1233.93 * invT);
    gRT[2] = lo[0] ? (fma(T, fma(T, fma(T, fma(T, 1.2532940000000001e-13, -5.807150833333333e-10), 1.059116e-06), -0.001737491), 0.7966090000000001) - 3.386842 * lnT + -30208.11 * invT) : (fma(T, fma(T, fma(T, fma(T, 3.195809e-16, -1.00083e-11), 1.4550433333333335e-07), -0.0015281465), -4.190671) - 2.672146 * lnT + -29899.21 * invT);
    if (hRT) hRT[2] = lo[0] ? (fma(T, fma(T, fma(T, fma(T, -5.013176000000001e-13, 1.74214525e-09), -2.118232e-06), 0.001737491), 3.386842) + -30208.11 * invT) : (fma(T, fma(T, fma(T, fma(T, -1.2783236e-15, 3.00249e-11), -2.910086666666667e-07), 0.0015281465), 2.672146) + -29899.21 * invT);
    gRT[3] = lo[0] ? (fma(T, fma(T, fma(T, fma(T, 0.0, 0.0), 0.0), 0.0), 2.9601176000000002) - 2.5 * lnT + 25471.63 * invT) : (fma(T, fma(T, fma(T, fma(T, 0.0, 0.0), 0.0), 0.0), 2.9601176000000002) - 2.5 * lnT + 25471.63 * invT);
    if (hRT) hRT[3] = lo[0] ? (fma(T, fma(T, fma(T, fma(T, 0.0, 0.0), 0.0), 0.0), 2.5) + 25471.63 * invT) : (fma(T, fma(T, fma(T, fma(T, 0.0, 0.0), 0.0), 0.0), 2.5) + 25471.63 * invT);
    gRT[4] = lo[0] ? (fma(T, fma(T, fma(T, fma(T, -1.945348e-14, 1.3357024999999999e-10), -4.035053333333333e-07), 0.000819083), -0.01756599999999997) - 2.946429 * lnT + 29147.64 * invT) : (fma(T, fma(T, fma(T, fma(T, 2.184026e-17, -3.7925558333333335e-13), 5.171338333333333e-10), 1.377531e-05), -2.378248) - 2.54206 * lnT + 29230.8 * invT);
    if (hRT) hRT[4] = lo[0] ? (fma(T, fma(T, fma(T, fma(T, 7.781392e-14, -4.0071075e-10), 8.070106666666666e-07), -0.000819083), 2.946429) + 29147.64 * invT) : (fma(T, fma(T, fma(T, fma(T, -8.736104e-17, 1.13776675e-12), -1.0342676666666666e-09), -1.377531e-05), 2.54206) + 29230.8 * invT);
    gRT[5] = lo[0] ? (fma(T, fma(T, fma(T, fma(T, -1.0311868949999999e-13, 4.832113691666666e-10), -1.0879411516666667e-06), 0.001612724695), 4.81573857) - 4.12530561 * lnT + 3346.30913 * invT) : (fma(T, fma(T, fma(T, fma(T, 6.6597938e-17, -2.54348895e-12), 4.318045966666667e-08), -0.00052825224), -2.8369118700000002) - 2.86472886 * lnT + 3683.62875 * invT);
    if (hRT) hRT[5] = lo[0] ? (fma(T, fma(T, fma(T, fma(T, 4.1247475799999997e-13, -1.4496341075e-09), 2.1758823033333334e-06), -0.001612724695), 4.12530561) + 3346.30913 * invT) : (fma(T, fma(T, fma(T, fma(T, -2.66391752e-16, 7.63046685e-12), -8.636091933333334e-08), 0.00052825224), 2.86472886) + 3683.62875 * invT);
    gRT[6] = lo[0] ? (fma(T, fma(T, fma(T, fma(T, -4.646125620000001e-13, 2.02303245e-09), -3.5263815166666663e-06), 0.002374560255), 0.5851355599999999) - 4.30179801 * lnT + 294.80804 * invT) : (fma(T, fma(T, fma(T, fma(T, 5.39542675e-16, -9.520530833333334e-12), 1.0560969166666666e-07), -0.001119910065), 0.23210875000000009) - 4.0172109 * lnT + 111.856713 * invT);
    if (hRT) hRT[6] = lo[0] ? (fma(T, fma(T, fma(T, fma(T, 1.8584502480000002e-12, -6.06909735e-09), 7.0527630333333326e-06), -0.002374560255), 4.30179801) + 294.80804 * invT) : (fma(T, fma(T, fma(T, fma(T, -2.1581707e-15, 2.85615925e-11), -2.1121938333333332e-07), 0.001119910065), 4.0172109) + 111.856713 * invT);
    gRT[7] = lo[0] ? (fma(T, fma(T, fma(T, fma(T, -1.2357574999999998e-13, 3.854838333333333e-10), 2.4750216666666664e-08), -0.003284613), -3.396609) - 3.388754 * lnT + -17663.15 * invT) : (fma(T, fma(T, fma(T, fma(T, 7.15827e-16, -1.9574199999999998e-11), 2.457815e-07), -0.002168068), 4.07203) - 4.573167 * lnT + -18006.96 * invT);
    if (hRT) hRT[7] = lo[0] ? (fma(T, fma(T, fma(T, fma(T, 4.943029999999999e-13, -1.1564515e-09), -4.950043333333333e-08), 0.003284613), 3.388754) + -17663.15 * invT) : (fma(T, fma(T, fma(T, fma(T, -2.863308e-15, 5.87226e-11), -4.91563e-07), 0.002168068), 4.573167) + -18006.96 * invT);
    gRT[8] = lo[0] ? (fma(T, fma(T, fma(T, fma(T, 1.2224275000000001e-13, -4.701262500000001e-10), 6.605369999999999e-07), -0.00070412), -0.6516950000000001) - 3.298677 * lnT + -1020.9 * invT) : (fma(T, fma(T, fma(T, fma(T, 3.3766754999999997e-16, -8.4142e-12), 9.474601666666666e-08), -0.0007439885), -3.0538879999999997) - 2.92664 * lnT + -922.7977 * invT);
    if (hRT) hRT[8] = lo[0] ? (fma(T, fma(T, fma(T, fma(T, -4.889710000000001e-13, 1.41037875e-09), -1.3210739999999999e-06), 0.00070412), 3.298677) + -1020.9 * invT) : (fma(T, fma(T, fma(T, fma(T, -1.3506701999999999e-15, 2.52426e-11), -1.8949203333333333e-07), 0.0007439885), 2.92664) + -922.7977 * invT);
  }
  // common T-dependent terms and per-species exp(g/RT) for reverse rates
  __host__ __device__ static inline void prelude(double T, double lnT, double invT, double* eg, double* hRT) {
    double gRT[9];
    g_h_RT(T, lnT, invT, gRT, hRT);
#pragma unroll
    for (int k = 0; k < 9; ++k) eg[k] = exp(gRT[k]);
  }
  // rates of progress q_j [mol/(cm^3 s)]; scale (may be null) multiplies each q_j
  template <bool MUL = false>
  __host__ __device__ static inline void progress(const double* C, double T, double* q, const double* rmul = nullptr) {
    RMUL_DEF;
    const double lnT = log(T), invT = 1.0 / T;
    const double refC = 0.012186596374704216 * invT, irefC = 82.05736608095968 * T;
    (void)refC; (void)irefC;
    double eg[9];
    prelude(T, lnT, invT, eg, nullptr);
    double ctot = 0.0;
#pragma unroll
    for (int k = 0; k < 9; ++k) ctot += C[k];
    const double M0 = ctot + 1.5 * C[0] + 11.0 * C[2];
    const double M1 = ctot + 1.0 * C[0] + -0.21999999999999997 * C[1] + 10.0 * C[2];
    {  // R0: H + O2 <=> O + OH
      const double kf = RMUL(exp(35.80487857070217 + -0.406 * lnT + -8352.941036546013 * invT), 0);
      const double Pf = C[1] * C[3];
      const double iKc = (eg[4] * eg[5]) / (eg[1] * eg[3]);
      const double Pb = C[4] * C[5];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      q[0] = qj;
    }
    {  // R1: O + H2 <=> H + OH
      const double kf = RMUL(exp(10.835651633566574 + 2.67 * lnT + -3165.2508657072367 * invT), 1);
      const double Pf = C[0] * C[4];
      const double iKc = (eg[3] * eg[5]) / (eg[0] * eg[4]);
      const double Pb = C[3] * C[5];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      q[1] = qj;
    }
    {  // R2: H2 + OH <=> H2O + H
      const double kf = RMUL(exp(19.19078896564844 + 1.51 * lnT + -1726.0429999007667 * invT), 2);
      const double Pf = C[0] * C[5];
      const double iKc = (eg[2] * eg[3]) / (eg[0] * eg[5]);
      const double Pb = C[2] * C[3];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      q[2] = qj;
    }
    {  // R3: O + H2O <=> OH + OH
      const double kf = RMUL(exp(14.904072510778882 + 2.02 * lnT + -6743.141748883461 * invT), 3);
      const double Pf = C[2] * C[4];
      const double iKc = (eg[5] * eg[5]) / (eg[2] * eg[4]);
      const double Pb = C[5] * C[5];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      q[3] = qj;
    }
    {  // R4: H2 + M <=> H + H + M
      const double kb = RMUL(exp(45.27016052855837 + -1.4 * lnT + -52526.05490660117 * invT), 4);
      const double kf = kb * M0;
      const double Pf = C[0];
      const double iKc = (eg[3] * eg[3] * irefC) / (eg[0]);
      const double Pb = C[3] * C[3];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      q[4] = qj;
    }
    {  // R5: O + O + M <=> O2 + M
      const double kb = RMUL(exp(36.35766453152699 + -0.5 * lnT), 5);
      const double kf = kb * M0;
      const double Pf = C[4] * C[4];
      const double iKc = (eg[1] * refC) / (eg[4] * eg[4]);
      const double Pb = C[1];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      q[5] = qj;
    }
    {  // R6: O + H + M <=> OH + M
      const double kb = RMUL((4.714e+18 * invT), 6);
      const double kf = kb * M0;
      const double Pf = C[3] * C[4];
      const double iKc = (eg[5] * refC) / (eg[3] * eg[4]);
      const double Pb = C[5];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      q[6] = qj;
    }
    {  // R7: H + OH + M <=> H2O + M
      const double kb = RMUL((3.8e+22 * invT*invT), 7);
      const double kf = kb * M0;
      const double Pf = C[3] * C[5];
      const double iKc = (eg[2] * refC) / (eg[3] * eg[5]);
      const double Pb = C[2];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      q[7] = qj;
    }
    {  // R8: H + O2 (+M) <=> HO2 (+M)
      const double kinf = exp(28.019679105720332 + 0.6 * lnT);
      const double Mj = M1;
      const double k0r = exp(19.88299408302048 + -2.32 * lnT + -264.08961118015225 * invT);
      const double Pr = fmax(k0r * Mj, 1e-300);
      const double iPr1 = 1.0 / (1.0 + Pr);
      const double lFc = -0.09691001300805639;
      const double cc = -0.33507029128460225, nn = 0.8730757165202316;
      const double xx = log10(Pr) + cc;
      const double DD = 1.0 / (nn - 0.14 * xx);
      const double f1 = xx * DD;
      const double iden = 1.0 / (1.0 + f1 * f1);
      const double F = exp(-0.22314355131420974 * iden);
      const double kf = RMUL(kinf * Pr * iPr1 * F, 8);
      const double Pf = C[1] * C[3];
      const double iKc = (eg[6] * refC) / (eg[1] * eg[3]);
      const double Pb = C[6];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      q[8] = qj;
    }
    {  // R9: HO2 + H <=> H2 + O2
      const double kf = RMUL(exp(30.440423811291044 + -414.14967606948426 * invT), 9);
      const double Pf = C[3] * C[6];
      const double iKc = (eg[0] * eg[1]) / (eg[3] * eg[6]);
      const double Pb = C[0] * C[1];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      q[9] = qj;
    }
    {  // R10: HO2 + H <=> OH + OH
      const double kf = RMUL(exp(31.890738863714645 + -148.4497623821359 * invT), 10);
      const double Pf = C[3] * C[6];
      const double iKc = (eg[5] * eg[5]) / (eg[3] * eg[6]);
      const double Pb = C[5] * C[5];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      q[10] = qj;
    }
    {  // R11: HO2 + O <=> O2 + OH
      const double kf = RMUL(32500000000000.0, 11);
      const double Pf = C[4] * C[6];
      const double iKc = (eg[1] * eg[5]) / (eg[4] * eg[6]);
      const double Pb = C[1] * C[5];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      q[11] = qj;
    }
    {  // R12: HO2 + OH <=> H2O + O2
      const double kf = RMUL(exp(30.994862711046935 + 250.1001081488866 * invT), 12);
      const double Pf = C[5] * C[6];
      const double iKc = (eg[1] * eg[2]) / (eg[5] * eg[6]);
      const double Pb = C[1] * C[2];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      q[12] = qj;
    }
    {  // R13: HO2 + HO2 <=> H2O2 + O2
      const double kf = RMUL(exp(33.67127582720596 + -6029.576450382212 * invT), 13);
      const double Pf = C[6] * C[6];
      const double iKc = (eg[1] * eg[7]) / (eg[6] * eg[6]);
      const double Pb = C[1] * C[7];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      q[13] = qj;
    }
    {  // R14: HO2 + HO2 <=> H2O2 + O2
      const double kf = RMUL(exp(25.590800287401994 + 819.895585929539 * invT), 14);
      const double Pf = C[6] * C[6];
      const double iKc = (eg[1] * eg[7]) / (eg[6] * eg[6]);
      const double Pb = C[1] * C[7];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      q[14] = qj;
    }
    {  // R15: H2O2 (+M) <=> OH + OH (+M)
      const double kinf = exp(33.31833539787744 + -24370.922007345227 * invT);
      const double Mj = M0;
      const double k0r = exp(6.009598019134351 + 0.0 * lnT + 1474.4332331513833 * invT);
      const double Pr = fmax(k0r * Mj, 1e-300);
      const double iPr1 = 1.0 / (1.0 + Pr);
      const double lFc = -0.3010299956639812;
      const double cc = -0.19830990290513262, nn = 1.1323080944932562;
      const double xx = log10(Pr) + cc;
      const double DD = 1.0 / (nn - 0.14 * xx);
      const double f1 = xx * DD;
      const double iden = 1.0 / (1.0 + f1 * f1);
      const double F = exp(-0.6931471805599454 * iden);
      const double kf = RMUL(kinf * Pr * iPr1 * F, 15);
      const double Pf = C[7];
      const double iKc = (eg[5] * eg[5] * irefC) / (eg[7]);
      const double Pb = C[5] * C[5];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      q[15] = qj;
    }
    {  // R16: H2O2 + H <=> H2O + OH
      const double kf = RMUL(exp(30.813232956425157 + -1997.7815479901 * invT), 16);
      const double Pf = C[3] * C[7];
      const double iKc = (eg[2] * eg[5]) / (eg[3] * eg[7]);
      const double Pb = C[2] * C[5];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      q[16] = qj;
    }
    {  // R17: H2O2 + H <=> HO2 + H2
      const double kf = RMUL(exp(31.506380136985104 + -4000.595291315188 * invT), 17);
      const double Pf = C[3] * C[7];
      const double iKc = (eg[0] * eg[6]) / (eg[3] * eg[7]);
      const double Pb = C[0] * C[6];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      q[17] = qj;
    }
    {  // R18: H2O2 + O <=> OH + HO2
      const double kf = RMUL(exp(16.07205171245691 + 2.0 * lnT + -1997.7815479901 * invT), 18);
      const double Pf = C[4] * C[7];
      const double iKc = (eg[5] * eg[6]) / (eg[4] * eg[7]);
      const double Pb = C[5] * C[6];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      q[18] = qj;
    }
    {  // R19: H2O2 + OH <=> HO2 + H2O
      const double kf = RMUL(1000000000000.0, 19);
      const double Pf = C[5] * C[7];
      const double iKc = (eg[2] * eg[6]) / (eg[5] * eg[7]);
      const double Pb = C[2] * C[6];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      q[19] = qj;
    }
    {  // R20: H2O2 + OH <=> HO2 + H2O
      const double kf = RMUL(exp(33.99404921946901 + -4809.269081647704 * invT), 20);
      const double Pf = C[5] * C[7];
      const double iKc = (eg[2] * eg[6]) / (eg[5] * eg[7]);
      const double Pb = C[2] * C[6];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      q[20] = qj;
    }
    {  // R21: 2 H + 2 OH => 2 H2O
      const double kf = RMUL(1e+27, 21);
      const double Pf = C[3] * C[3] * C[5] * C[5];
      const double net = Pf;
      const double qj = kf * net;
      q[21] = qj;
    }
  }
  // molar production rates wdot_k [mol/(cm^3 s)]
  template <bool MUL = false>
  __host__ __device__ static inline void wdot(const double* C, double T, double* wd, const double* rmul = nullptr) {
    RMUL_DEF;
    double lnT = log(T), invT = 1.0 / T;
    const double refC = 0.012186596374704216 * invT, irefC = 82.05736608095968 * T;
    (void)refC; (void)irefC;
    double eg[9];
    prelude(T, lnT, invT, eg, nullptr);
    double ctot = 0.0;
#pragma unroll
    for (int k = 0; k < 9; ++k) ctot += C[k];
    const double M0 = ctot + 1.5 * C[0] + 11.0 * C[2];
    const double M1 = ctot + 1.0 * C[0] + -0.21999999999999997 * C[1] + 10.0 * C[2];
#pragma unroll
    for (int k = 0; k < 9; ++k) wd[k] = 0.0;
    {  // R0: H + O2 <=> O + OH
      const double kf = RMUL(exp(35.80487857070217 + -0.406 * lnT + -8352.941036546013 * invT), 0);
      const double Pf = C[1] * C[3];
      const double iKc = (eg[4] * eg[5]) / (eg[1] * eg[3]);
      const double Pb = C[4] * C[5];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      wd[1] += -1.0 * qj;
      wd[3] += -1.0 * qj;
      wd[4] += 1.0 * qj;
      wd[5] += 1.0 * qj;
    }
    {  // R1: O + H2 <=> H + OH
      const double kf = RMUL(exp(10.835651633566574 + 2.67 * lnT + -3165.2508657072367 * invT), 1);
      const double Pf = C[0] * C[4];
      const double iKc = (eg[3] * eg[5]) / (eg[0] * eg[4]);
      const double Pb = C[3] * C[5];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      wd[0] += -1.0 * qj;
      wd[3] += 1.0 * qj;
      wd[4] += -1.0 * qj;
      wd[5] += 1.0 * qj;
    }
    {  // R2: H2 + OH <=> H2O + H
      const double kf = RMUL(exp(19.19078896564844 + 1.51 * lnT + -1726.0429999007667 * invT), 2);
      const double Pf = C[0] * C[5];
      const double iKc = (eg[2] * eg[3]) / (eg[0] * eg[5]);
      const double Pb = C[2] * C[3];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      wd[0] += -1.0 * qj;
      wd[2] += 1.0 * qj;
      wd[3] += 1.0 * qj;
      wd[5] += -1.0 * qj;
    }
    {  // R3: O + H2O <=> OH + OH
      const double kf = RMUL(exp(14.904072510778882 + 2.02 * lnT + -6743.141748883461 * invT), 3);
      const double Pf = C[2] * C[4];
      const double iKc = (eg[5] * eg[5]) / (eg[2] * eg[4]);
      const double Pb = C[5] * C[5];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      wd[2] += -1.0 * qj;
      wd[4] += -1.0 * qj;
      wd[5] += 2.0 * qj;
    }
    {  // R4: H2 + M <=> H + H + M
      const double kb = RMUL(exp(45.27016052855837 + -1.4 * lnT + -52526.05490660117 * invT), 4);
      const double kf = kb * M0;
      const double Pf = C[0];
      const double iKc = (eg[3] * eg[3] * irefC) / (eg[0]);
      const double Pb = C[3] * C[3];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      wd[0] += -1.0 * qj;
      wd[3] += 2.0 * qj;
    }
    {  // R5: O + O + M <=> O2 + M
      const double kb = RMUL(exp(36.35766453152699 + -0.5 * lnT), 5);
      const double kf = kb * M0;
      const double Pf = C[4] * C[4];
      const double iKc = (eg[1] * refC) / (eg[4] * eg[4]);
      const double Pb = C[1];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      wd[1] += 1.0 * qj;
      wd[4] += -2.0 * qj;
    }
    {  // R6: O + H + M <=> OH + M
      const double kb = RMUL((4.714e+18 * invT), 6);
      const double kf = kb * M0;
      const double Pf = C[3] * C[4];
      const double iKc = (eg[5] * refC) / (eg[3] * eg[4]);
      const double Pb = C[5];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      wd[3] += -1.0 * qj;
      wd[4] += -1.0 * qj;
      wd[5] += 1.0 * qj;
    }
    {  // R7: H + OH + M <=> H2O + M
      const double kb = RMUL((3.8e+22 * invT*invT), 7);
      const double kf = kb * M0;
      const double Pf = C[3] * C[5];
      const double iKc = (eg[2] * refC) / (eg[3] * eg[5]);
      const double Pb = C[2];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      wd[2] += 1.0 * qj;
      wd[3] += -1.0 * qj;
      wd[5] += -1.0 * qj;
    }
    {  // R8: H + O2 (+M) <=> HO2 (+M)
      const double kinf = exp(28.019679105720332 + 0.6 * lnT);
      const double Mj = M1;
      const double k0r = exp(19.88299408302048 + -2.32 * lnT + -264.08961118015225 * invT);
      const double Pr = fmax(k0r * Mj, 1e-300);
      const double iPr1 = 1.0 / (1.0 + Pr);
      const double lFc = -0.09691001300805639;
      const double cc = -0.33507029128460225, nn = 0.8730757165202316;
      const double xx = log10(Pr) + cc;
      const double DD = 1.0 / (nn - 0.14 * xx);
      const double f1 = xx * DD;
      const double iden = 1.0 / (1.0 + f1 * f1);
      const double F = exp(-0.22314355131420974 * iden);
      const double kf = RMUL(kinf * Pr * iPr1 * F, 8);
      const double Pf = C[1] * C[3];
      const double iKc = (eg[6] * refC) / (eg[1] * eg[3]);
      const double Pb = C[6];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      wd[1] += -1.0 * qj;
      wd[3] += -1.0 * qj;
      wd[6] += 1.0 * qj;
    }
    {  // R9: HO2 + H <=> H2 + O2
      const double kf = RMUL(exp(30.440423811291044 + -414.14967606948426 * invT), 9);
      const double Pf = C[3] * C[6];
      const double iKc = (eg[0] * eg[1]) / (eg[3] * eg[6]);
      const double Pb = C[0] * C[1];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      wd[0] += 1.0 * qj;
      wd[1] += 1.0 * qj;
      wd[3] += -1.0 * qj;
      wd[6] += -1.0 * qj;
    }
    {  // R10: HO2 + H <=> OH + OH
      const double kf = RMUL(exp(31.890738863714645 + -148.4497623821359 * invT), 10);
      const double Pf = C[3] * C[6];
      const double iKc = (eg[5] * eg[5]) / (eg[3] * eg[6]);
      const double Pb = C[5] * C[5];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      wd[3] += -1.0 * qj;
      wd[5] += 2.0 * qj;
      wd[6] += -1.0 * qj;
    }
    {  // R11: HO2 + O <=> O2 + OH
      const double kf = RMUL(32500000000000.0, 11);
      const double Pf = C[4] * C[6];
      const double iKc = (eg[1] * eg[5]) / (eg[4] * eg[6]);
      const double Pb = C[1] * C[5];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      wd[1] += 1.0 * qj;
      wd[4] += -1.0 * qj;
      wd[5] += 1.0 * qj;
      wd[6] += -1.0 * qj;
    }
    {  // R12: HO2 + OH <=> H2O + O2
      const double kf = RMUL(exp(30.994862711046935 + 250.1001081488866 * invT), 12);
      const double Pf = C[5] * C[6];
      const double iKc = (eg[1] * eg[2]) / (eg[5] * eg[6]);
      const double Pb = C[1] * C[2];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      wd[1] += 1.0 * qj;
      wd[2] += 1.0 * qj;
      wd[5] += -1.0 * qj;
      wd[6] += -1.0 * qj;
    }
    {  // R13: HO2 + HO2 <=> H2O2 + O2
      const double kf = RMUL(exp(33.67127582720596 + -6029.576450382212 * invT), 13);
      const double Pf = C[6] * C[6];
      const double iKc = (eg[1] * eg[7]) / (eg[6] * eg[6]);
      const double Pb = C[1] * C[7];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      wd[1] += 1.0 * qj;
      wd[6] += -2.0 * qj;
      wd[7] += 1.0 * qj;
    }
    {  // R14: HO2 + HO2 <=> H2O2 + O2
      const double kf = RMUL(exp(25.590800287401994 + 819.895585929539 * invT), 14);
      const double Pf = C[6] * C[6];
      const double iKc = (eg[1] * eg[7]) / (eg[6] * eg[6]);
      const double Pb = C[1] * C[7];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      wd[1] += 1.0 * qj;
      wd[6] += -2.0 * qj;
      wd[7] += 1.0 * qj;
    }
    {  // R15: H2O2 (+M) <=> OH + OH (+M)
      const double kinf = exp(33.31833539787744 + -24370.922007345227 * invT);
      const double Mj = M0;
      const double k0r = exp(6.009598019134351 + 0.0 * lnT + 1474.4332331513833 * invT);
      const double Pr = fmax(k0r * Mj, 1e-300);
      const double iPr1 = 1.0 / (1.0 + Pr);
      const double lFc = -0.3010299956639812;
      const double cc = -0.19830990290513262, nn = 1.1323080944932562;
      const double xx = log10(Pr) + cc;
      const double DD = 1.0 / (nn - 0.14 * xx);
      const double f1 = xx * DD;
      const double iden = 1.0 / (1.0 + f1 * f1);
      const double F = exp(-0.6931471805599454 * iden);
      const double kf = RMUL(kinf * Pr * iPr1 * F, 15);
      const double Pf = C[7];
      const double iKc = (eg[5] * eg[5] * irefC) / (eg[7]);
      const double Pb = C[5] * C[5];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      wd[5] += 2.0 * qj;
      wd[7] += -1.0 * qj;
    }
    {  // R16: H2O2 + H <=> H2O + OH
      const double kf = RMUL(exp(30.813232956425157 + -1997.7815479901 * invT), 16);
      const double Pf = C[3] * C[7];
      const double iKc = (eg[2] * eg[5]) / (eg[3] * eg[7]);
      const double Pb = C[2] * C[5];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      wd[2] += 1.0 * qj;
      wd[3] += -1.0 * qj;
      wd[5] += 1.0 * qj;
      wd[7] += -1.0 * qj;
    }
    {  // R17: H2O2 + H <=> HO2 + H2
      const double kf = RMUL(exp(31.506380136985104 + -4000.595291315188 * invT), 17);
      const double Pf = C[3] * C[7];
      const double iKc = (eg[0] * eg[6]) / (eg[3] * eg[7]);
      const double Pb = C[0] * C[6];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      wd[0] += 1.0 * qj;
      wd[3] += -1.0 * qj;
      wd[6] += 1.0 * qj;
      wd[7] += -1.0 * qj;
    }
    {  // R18: H2O2 + O <=> OH + HO2
      const double kf = RMUL(exp(16.07205171245691 + 2.0 * lnT + -1997.7815479901 * invT), 18);
      const double Pf = C[4] * C[7];
      const double iKc = (eg[5] * eg[6]) / (eg[4] * eg[7]);
      const double Pb = C[5] * C[6];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      wd[4] += -1.0 * qj;
      wd[5] += 1.0 * qj;
      wd[6] += 1.0 * qj;
      wd[7] += -1.0 * qj;
    }
    {  // R19: H2O2 + OH <=> HO2 + H2O
      const double kf = RMUL(1000000000000.0, 19);
      const double Pf = C[5] * C[7];
      const double iKc = (eg[2] * eg[6]) / (eg[5] * eg[7]);
      const double Pb = C[2] * C[6];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      wd[2] += 1.0 * qj;
      wd[5] += -1.0 * qj;
      wd[6] += 1.0 * qj;
      wd[7] += -1.0 * qj;
    }
    {  // R20: H2O2 + OH <=> HO2 + H2O
      const double kf = RMUL(exp(33.99404921946901 + -4809.269081647704 * invT), 20);
      const double Pf = C[5] * C[7];
      const double iKc = (eg[2] * eg[6]) / (eg[5] * eg[7]);
      const double Pb = C[2] * C[6];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      wd[2] += 1.0 * qj;
      wd[5] += -1.0 * qj;
      wd[6] += 1.0 * qj;
      wd[7] += -1.0 * qj;
    }
    {  // R21: 2 H + 2 OH => 2 H2O
      const double kf = RMUL(1e+27, 21);
      const double Pf = C[3] * C[3] * C[5] * C[5];
      const double net = Pf;
      const double qj = kf * net;
      wd[2] += 2.0 * qj;
      wd[3] += -2.0 * qj;
      wd[5] += -2.0 * qj;
    }
  }
  // wdot and its Jacobian: dwdC[k*LD+m] = d wdot_k / d C_m, dwdT[k] = d wdot_k / dT
  template <int LD, typename JT, bool MUL = false>
  __host__ __device__ static inline void wdot_jac(const double* C, double T, double* wd, JT* dwdC, double* dwdT, const double* rmul = nullptr) {
    RMUL_DEF;
    double lnT = log(T), invT = 1.0 / T;
    const double refC = 0.012186596374704216 * invT, irefC = 82.05736608095968 * T;
    (void)refC; (void)irefC;
    double eg[9], hRT[9];
    prelude(T, lnT, invT, eg, hRT);
    double ctot = 0.0;
#pragma unroll
    for (int k = 0; k < 9; ++k) ctot += C[k];
    const double M0 = ctot + 1.5 * C[0] + 11.0 * C[2];
    const double M1 = ctot + 1.0 * C[0] + -0.21999999999999997 * C[1] + 10.0 * C[2];
#pragma unroll
    for (int k = 0; k < 9; ++k) { wd[k] = 0.0; dwdT[k] = 0.0; }
#pragma unroll
    for (int k = 0; k < 9; ++k)
#pragma unroll
      for (int m = 0; m < 9; ++m) dwdC[k * LD + m] = JT(0);
    {  // R0: H + O2 <=> O + OH
      const double kf = RMUL(exp(35.80487857070217 + -0.406 * lnT + -8352.941036546013 * invT), 0);
      const double dlnk = (-0.406 + 8352.941036546013 * invT) * invT;
      const double Pf = C[1] * C[3];
      const double iKc = (eg[4] * eg[5]) / (eg[1] * eg[3]);
      const double Pb = C[4] * C[5];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      const double dlnKc = (-1.0 * hRT[1] + -1.0 * hRT[3] + 1.0 * hRT[4] + 1.0 * hRT[5] - 0.0) * invT;
      const double dqdT = kf * (dlnk * net + iKc * Pb * dlnKc);
      const double dq1 = kf * (C[3]);
      const double dq3 = kf * (C[1]);
      const double dq4 = -kf * iKc * (C[5]);
      const double dq5 = -kf * iKc * (C[4]);
      wd[1] += -1.0 * qj;
      dwdT[1] += -1.0 * dqdT;
      dwdC[1 * LD + 1] += JT(-1.0 * dq1);
      dwdC[1 * LD + 3] += JT(-1.0 * dq3);
      dwdC[1 * LD + 4] += JT(-1.0 * dq4);
      dwdC[1 * LD + 5] += JT(-1.0 * dq5);
      wd[3] += -1.0 * qj;
      dwdT[3] += -1.0 * dqdT;
      dwdC[3 * LD + 1] += JT(-1.0 * dq1);
      dwdC[3 * LD + 3] += JT(-1.0 * dq3);
      dwdC[3 * LD + 4] += JT(-1.0 * dq4);
      dwdC[3 * LD + 5] += JT(-1.0 * dq5);
      wd[4] += 1.0 * qj;
      dwdT[4] += 1.0 * dqdT;
      dwdC[4 * LD + 1] += JT(1.0 * dq1);
      dwdC[4 * LD + 3] += JT(1.0 * dq3);
      dwdC[4 * LD + 4] += JT(1.0 * dq4);
      dwdC[4 * LD + 5] += JT(1.0 * dq5);
      wd[5] += 1.0 * qj;
      dwdT[5] += 1.0 * dqdT;
      dwdC[5 * LD + 1] += JT(1.0 * dq1);
      dwdC[5 * LD + 3] += JT(1.0 * dq3);
      dwdC[5 * LD + 4] += JT(1.0 * dq4);
      dwdC[5 * LD + 5] += JT(1.0 * dq5);
      PELEC_MEMORY_FENCE();
    }
    {  // R1: O + H2 <=> H + OH
      const double kf = RMUL(exp(10.835651633566574 + 2.67 * lnT + -3165.2508657072367 * invT), 1);
      const double dlnk = (2.67 + 3165.2508657072367 * invT) * invT;
      const double Pf = C[0] * C[4];
      const double iKc = (eg[3] * eg[5]) / (eg[0] * eg[4]);
      const double Pb = C[3] * C[5];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      const double dlnKc = (-1.0 * hRT[0] + 1.0 * hRT[3] + -1.0 * hRT[4] + 1.0 * hRT[5] - 0.0) * invT;
      const double dqdT = kf * (dlnk * net + iKc * Pb * dlnKc);
      const double dq0 = kf * (C[4]);
      const double dq3 = -kf * iKc * (C[5]);
      const double dq4 = kf * (C[0]);
      const double dq5 = -kf * iKc * (C[3]);
      wd[0] += -1.0 * qj;
      dwdT[0] += -1.0 * dqdT;
      dwdC[0 * LD + 0] += JT(-1.0 * dq0);
      dwdC[0 * LD + 3] += JT(-1.0 * dq3);
      dwdC[0 * LD + 4] += JT(-1.0 * dq4);
      dwdC[0 * LD + 5] += JT(-1.0 * dq5);
      wd[3] += 1.0 * qj;
      dwdT[3] += 1.0 * dqdT;
      dwdC[3 * LD + 0] += JT(1.0 * dq0);
      dwdC[3 * LD + 3] += JT(1.0 * dq3);
      dwdC[3 * LD + 4] += JT(1.0 * dq4);
      dwdC[3 * LD + 5] += JT(1.0 * dq5);
      wd[4] += -1.0 * qj;
      dwdT[4] += -1.0 * dqdT;
      dwdC[4 * LD + 0] += JT(-1.0 * dq0);
      dwdC[4 * LD + 3] += JT(-1.0 * dq3);
      dwdC[4 * LD + 4] += JT(-1.0 * dq4);
      dwdC[4 * LD + 5] += JT(-1.0 * dq5);
      wd[5] += 1.0 * qj;
      dwdT[5] += 1.0 * dqdT;
      dwdC[5 * LD + 0] += JT(1.0 * dq0);
      dwdC[5 * LD + 3] += JT(1.0 * dq3);
      dwdC[5 * LD + 4] += JT(1.0 * dq4);
      dwdC[5 * LD + 5] += JT(1.0 * dq5);
      PELEC_MEMORY_FENCE();
    }
    {  // R2: H2 + OH <=> H2O + H
      const double kf = RMUL(exp(19.19078896564844 + 1.51 * lnT + -1726.0429999007667 * invT), 2);
      const double dlnk = (1.51 + 1726.0429999007667 * invT) * invT;
      const double Pf = C[0] * C[5];
      const double iKc = (eg[2] * eg[3]) / (eg[0] * eg[5]);
      const double Pb = C[2] * C[3];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      const double dlnKc = (-1.0 * hRT[0] + 1.0 * hRT[2] + 1.0 * hRT[3] + -1.0 * hRT[5] - 0.0) * invT;
      const double dqdT = kf * (dlnk * net + iKc * Pb * dlnKc);
      const double dq0 = kf * (C[5]);
      const double dq2 = -kf * iKc * (C[3]);
      const double dq3 = -kf * iKc * (C[2]);
      const double dq5 = kf * (C[0]);
      wd[0] += -1.0 * qj;
      dwdT[0] += -1.0 * dqdT;
      dwdC[0 * LD + 0] += JT(-1.0 * dq0);
      dwdC[0 * LD + 2] += JT(-1.0 * dq2);
      dwdC[0 * LD + 3] += JT(-1.0 * dq3);
      dwdC[0 * LD + 5] += JT(-1.0 * dq5);
      wd[2] += 1.0 * qj;
      dwdT[2] += 1.0 * dqdT;
      dwdC[2 * LD + 0] += JT(1.0 * dq0);
      dwdC[2 * LD + 2] += JT(1.0 * dq2);
      dwdC[2 * LD + 3] += JT(1.0 * dq3);
      dwdC[2 * LD + 5] += JT(1.0 * dq5);
      wd[3] += 1.0 * qj;
      dwdT[3] += 1.0 * dqdT;
      dwdC[3 * LD + 0] += JT(1.0 * dq0);
      dwdC[3 * LD + 2] += JT(1.0 * dq2);
      dwdC[3 * LD + 3] += JT(1.0 * dq3);
      dwdC[3 * LD + 5] += JT(1.0 * dq5);
      wd[5] += -1.0 * qj;
      dwdT[5] += -1.0 * dqdT;
      dwdC[5 * LD + 0] += JT(-1.0 * dq0);
      dwdC[5 * LD + 2] += JT(-1.0 * dq2);
      dwdC[5 * LD + 3] += JT(-1.0 * dq3);
      dwdC[5 * LD + 5] += JT(-1.0 * dq5);
      PELEC_MEMORY_FENCE();
    }
    {  // R3: O + H2O <=> OH + OH
      const double kf = RMUL(exp(14.904072510778882 + 2.02 * lnT + -6743.141748883461 * invT), 3);
      const double dlnk = (2.02 + 6743.141748883461 * invT) * invT;
      const double Pf = C[2] * C[4];
      const double iKc = (eg[5] * eg[5]) / (eg[2] * eg[4]);
      const double Pb = C[5] * C[5];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      const double dlnKc = (-1.0 * hRT[2] + -1.0 * hRT[4] + 2.0 * hRT[5] - 0.0) * invT;
      const double dqdT = kf * (dlnk * net + iKc * Pb * dlnKc);
      const double dq2 = kf * (C[4]);
      const double dq4 = kf * (C[2]);
      const double dq5 = -kf * iKc * (2.0 * C[5]);
      wd[2] += -1.0 * qj;
      dwdT[2] += -1.0 * dqdT;
      dwdC[2 * LD + 2] += JT(-1.0 * dq2);
      dwdC[2 * LD + 4] += JT(-1.0 * dq4);
      dwdC[2 * LD + 5] += JT(-1.0 * dq5);
      wd[4] += -1.0 * qj;
      dwdT[4] += -1.0 * dqdT;
      dwdC[4 * LD + 2] += JT(-1.0 * dq2);
      dwdC[4 * LD + 4] += JT(-1.0 * dq4);
      dwdC[4 * LD + 5] += JT(-1.0 * dq5);
      wd[5] += 2.0 * qj;
      dwdT[5] += 2.0 * dqdT;
      dwdC[5 * LD + 2] += JT(2.0 * dq2);
      dwdC[5 * LD + 4] += JT(2.0 * dq4);
      dwdC[5 * LD + 5] += JT(2.0 * dq5);
      PELEC_MEMORY_FENCE();
    }
    {  // R4: H2 + M <=> H + H + M
      const double kb = RMUL(exp(45.27016052855837 + -1.4 * lnT + -52526.05490660117 * invT), 4);
      const double kf = kb * M0;
      const double dkdM = kb;
      const double dlnk = (-1.4 + 52526.05490660117 * invT) * invT;
      const double Pf = C[0];
      const double iKc = (eg[3] * eg[3] * irefC) / (eg[0]);
      const double Pb = C[3] * C[3];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      const double dlnKc = (-1.0 * hRT[0] + 2.0 * hRT[3] - 1.0) * invT;
      const double dqdT = kf * (dlnk * net + iKc * Pb * dlnKc);
      const double dq0 = kf * (1.0);
      const double dq3 = -kf * iKc * (2.0 * C[3]);
      wd[0] += -1.0 * qj;
      dwdT[0] += -1.0 * dqdT;
      dwdC[0 * LD + 0] += JT(-1.0 * dq0);
      dwdC[0 * LD + 3] += JT(-1.0 * dq3);
      wd[3] += 2.0 * qj;
      dwdT[3] += 2.0 * dqdT;
      dwdC[3 * LD + 0] += JT(2.0 * dq0);
      dwdC[3 * LD + 3] += JT(2.0 * dq3);
      const double dqdM = dkdM * net;
      dwdC[0 * LD + 0] += JT(-2.5 * dqdM);
      dwdC[0 * LD + 1] += JT(-1.0 * dqdM);
      dwdC[0 * LD + 2] += JT(-12.0 * dqdM);
      dwdC[0 * LD + 3] += JT(-1.0 * dqdM);
      dwdC[0 * LD + 4] += JT(-1.0 * dqdM);
      dwdC[0 * LD + 5] += JT(-1.0 * dqdM);
      dwdC[0 * LD + 6] += JT(-1.0 * dqdM);
      dwdC[0 * LD + 7] += JT(-1.0 * dqdM);
      dwdC[0 * LD + 8] += JT(-1.0 * dqdM);
      dwdC[3 * LD + 0] += JT(5.0 * dqdM);
      dwdC[3 * LD + 1] += JT(2.0 * dqdM);
      dwdC[3 * LD + 2] += JT(24.0 * dqdM);
      dwdC[3 * LD + 3] += JT(2.0 * dqdM);
      dwdC[3 * LD + 4] += JT(2.0 * dqdM);
      dwdC[3 * LD + 5] += JT(2.0 * dqdM);
      dwdC[3 * LD + 6] += JT(2.0 * dqdM);
      dwdC[3 * LD + 7] += JT(2.0 * dqdM);
      dwdC[3 * LD + 8] += JT(2.0 * dqdM);
      PELEC_MEMORY_FENCE();
    }
    {  // R5: O + O + M <=> O2 + M
      const double kb = RMUL(exp(36.35766453152699 + -0.5 * lnT), 5);
      const double kf = kb * M0;
      const double dkdM = kb;
      const double dlnk = (-0.5 + 0.0 * invT) * invT;
      const double Pf = C[4] * C[4];
      const double iKc = (eg[1] * refC) / (eg[4] * eg[4]);
      const double Pb = C[1];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      const double dlnKc = (1.0 * hRT[1] + -2.0 * hRT[4] - -1.0) * invT;
      const double dqdT = kf * (dlnk * net + iKc * Pb * dlnKc);
      const double dq1 = -kf * iKc * (1.0);
      const double dq4 = kf * (2.0 * C[4]);
      wd[1] += 1.0 * qj;
      dwdT[1] += 1.0 * dqdT;
      dwdC[1 * LD + 1] += JT(1.0 * dq1);
      dwdC[1 * LD + 4] += JT(1.0 * dq4);
      wd[4] += -2.0 * qj;
      dwdT[4] += -2.0 * dqdT;
      dwdC[4 * LD + 1] += JT(-2.0 * dq1);
      dwdC[4 * LD + 4] += JT(-2.0 * dq4);
      const double dqdM = dkdM * net;
      dwdC[1 * LD + 0] += JT(2.5 * dqdM);
      dwdC[1 * LD + 1] += JT(1.0 * dqdM);
      dwdC[1 * LD + 2] += JT(12.0 * dqdM);
      dwdC[1 * LD + 3] += JT(1.0 * dqdM);
      dwdC[1 * LD + 4] += JT(1.0 * dqdM);
      dwdC[1 * LD + 5] += JT(1.0 * dqdM);
      dwdC[1 * LD + 6] += JT(1.0 * dqdM);
      dwdC[1 * LD + 7] += JT(1.0 * dqdM);
      dwdC[1 * LD + 8] += JT(1.0 * dqdM);
      dwdC[4 * LD + 0] += JT(-5.0 * dqdM);
      dwdC[4 * LD + 1] += JT(-2.0 * dqdM);
      dwdC[4 * LD + 2] += JT(-24.0 * dqdM);
      dwdC[4 * LD + 3] += JT(-2.0 * dqdM);
      dwdC[4 * LD + 4] += JT(-2.0 * dqdM);
      dwdC[4 * LD + 5] += JT(-2.0 * dqdM);
      dwdC[4 * LD + 6] += JT(-2.0 * dqdM);
      dwdC[4 * LD + 7] += JT(-2.0 * dqdM);
      dwdC[4 * LD + 8] += JT(-2.0 * dqdM);
      PELEC_MEMORY_FENCE();
    }
    {  // R6: O + H + M <=> OH + M
      const double kb = RMUL((4.714e+18 * invT), 6);
      const double kf = kb * M0;
      const double dkdM = kb;
      const double dlnk = (-1.0 + 0.0 * invT) * invT;
      const double Pf = C[3] * C[4];
      const double iKc = (eg[5] * refC) / (eg[3] * eg[4]);
      const double Pb = C[5];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      const double dlnKc = (-1.0 * hRT[3] + -1.0 * hRT[4] + 1.0 * hRT[5] - -1.0) * invT;
      const double dqdT = kf * (dlnk * net + iKc * Pb * dlnKc);
      const double dq3 = kf * (C[4]);
      const double dq4 = kf * (C[3]);
      const double dq5 = -kf * iKc * (1.0);
      wd[3] += -1.0 * qj;
      dwdT[3] += -1.0 * dqdT;
      dwdC[3 * LD + 3] += JT(-1.0 * dq3);
      dwdC[3 * LD + 4] += JT(-1.0 * dq4);
      dwdC[3 * LD + 5] += JT(-1.0 * dq5);
      wd[4] += -1.0 * qj;
      dwdT[4] += -1.0 * dqdT;
      dwdC[4 * LD + 3] += JT(-1.0 * dq3);
      dwdC[4 * LD + 4] += JT(-1.0 * dq4);
      dwdC[4 * LD + 5] += JT(-1.0 * dq5);
      wd[5] += 1.0 * qj;
      dwdT[5] += 1.0 * dqdT;
      dwdC[5 * LD + 3] += JT(1.0 * dq3);
      dwdC[5 * LD + 4] += JT(1.0 * dq4);
      dwdC[5 * LD + 5] += JT(1.0 * dq5);
      const double dqdM = dkdM * net;
      dwdC[3 * LD + 0] += JT(-2.5 * dqdM);
      dwdC[3 * LD + 1] += JT(-1.0 * dqdM);
      dwdC[3 * LD + 2] += JT(-12.0 * dqdM);
      dwdC[3 * LD + 3] += JT(-1.0 * dqdM);
      dwdC[3 * LD + 4] += JT(-1.0 * dqdM);
      dwdC[3 * LD + 5] += JT(-1.0 * dqdM);
      dwdC[3 * LD + 6] += JT(-1.0 * dqdM);
      dwdC[3 * LD + 7] += JT(-1.0 * dqdM);
      dwdC[3 * LD + 8] += JT(-1.0 * dqdM);
      dwdC[4 * LD + 0] += JT(-2.5 * dqdM);
      dwdC[4 * LD + 1] += JT(-1.0 * dqdM);
      dwdC[4 * LD + 2] += JT(-12.0 * dqdM);
      dwdC[4 * LD + 3] += JT(-1.0 * dqdM);
      dwdC[4 * LD + 4] += JT(-1.0 * dqdM);
      dwdC[4 * LD + 5] += JT(-1.0 * dqdM);
      dwdC[4 * LD + 6] += JT(-1.0 * dqdM);
      dwdC[4 * LD + 7] += JT(-1.0 * dqdM);
      dwdC[4 * LD + 8] += JT(-1.0 * dqdM);
      dwdC[5 * LD + 0] += JT(2.5 * dqdM);
      dwdC[5 * LD + 1] += JT(1.0 * dqdM);
      dwdC[5 * LD + 2] += JT(12.0 * dqdM);
      dwdC[5 * LD + 3] += JT(1.0 * dqdM);
      dwdC[5 * LD + 4] += JT(1.0 * dqdM);
      dwdC[5 * LD + 5] += JT(1.0 * dqdM);
      dwdC[5 * LD + 6] += JT(1.0 * dqdM);
      dwdC[5 * LD + 7] += JT(1.0 * dqdM);
      dwdC[5 * LD + 8] += JT(1.0 * dqdM);
      PELEC_MEMORY_FENCE();
    }
    {  // R7: H + OH + M <=> H2O + M
      const double kb = RMUL((3.8e+22 * invT*invT), 7);
      const double kf = kb * M0;
      const double dkdM = kb;
      const double dlnk = (-2.0 + 0.0 * invT) * invT;
      const double Pf = C[3] * C[5];
      const double iKc = (eg[2] * refC) / (eg[3] * eg[5]);
      const double Pb = C[2];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      const double dlnKc = (1.0 * hRT[2] + -1.0 * hRT[3] + -1.0 * hRT[5] - -1.0) * invT;
      const double dqdT = kf * (dlnk * net + iKc * Pb * dlnKc);
      const double dq2 = -kf * iKc * (1.0);
      const double dq3 = kf * (C[5]);
      const double dq5 = kf * (C[3]);
      wd[2] += 1.0 * qj;
      dwdT[2] += 1.0 * dqdT;
      dwdC[2 * LD + 2] += JT(1.0 * dq2);
      dwdC[2 * LD + 3] += JT(1.0 * dq3);
      dwdC[2 * LD + 5] += JT(1.0 * dq5);
      wd[3] += -1.0 * qj;
      dwdT[3] += -1.0 * dqdT;
      dwdC[3 * LD + 2] += JT(-1.0 * dq2);
      dwdC[3 * LD + 3] += JT(-1.0 * dq3);
      dwdC[3 * LD + 5] += JT(-1.0 * dq5);
      wd[5] += -1.0 * qj;
      dwdT[5] += -1.0 * dqdT;
      dwdC[5 * LD + 2] += JT(-1.0 * dq2);
      dwdC[5 * LD + 3] += JT(-1.0 * dq3);
      dwdC[5 * LD + 5] += JT(-1.0 * dq5);
      const double dqdM = dkdM * net;
      dwdC[2 * LD + 0] += JT(2.5 * dqdM);
      dwdC[2 * LD + 1] += JT(1.0 * dqdM);
      dwdC[2 * LD + 2] += JT(12.0 * dqdM);
      dwdC[2 * LD + 3] += JT(1.0 * dqdM);
      dwdC[2 * LD + 4] += JT(1.0 * dqdM);
      dwdC[2 * LD + 5] += JT(1.0 * dqdM);
      dwdC[2 * LD + 6] += JT(1.0 * dqdM);
      dwdC[2 * LD + 7] += JT(1.0 * dqdM);
      dwdC[2 * LD + 8] += JT(1.0 * dqdM);
      dwdC[3 * LD + 0] += JT(-2.5 * dqdM);
      dwdC[3 * LD + 1] += JT(-1.0 * dqdM);
      dwdC[3 * LD + 2] += JT(-12.0 * dqdM);
      dwdC[3 * LD + 3] += JT(-1.0 * dqdM);
      dwdC[3 * LD + 4] += JT(-1.0 * dqdM);
      dwdC[3 * LD + 5] += JT(-1.0 * dqdM);
      dwdC[3 * LD + 6] += JT(-1.0 * dqdM);
      dwdC[3 * LD + 7] += JT(-1.0 * dqdM);
      dwdC[3 * LD + 8] += JT(-1.0 * dqdM);
      dwdC[5 * LD + 0] += JT(-2.5 * dqdM);
      dwdC[5 * LD + 1] += JT(-1.0 * dqdM);
      dwdC[5 * LD + 2] += JT(-12.0 * dqdM);
      dwdC[5 * LD + 3] += JT(-1.0 * dqdM);
      dwdC[5 * LD + 4] += JT(-1.0 * dqdM);
      dwdC[5 * LD + 5] += JT(-1.0 * dqdM);
      dwdC[5 * LD + 6] += JT(-1.0 * dqdM);
      dwdC[5 * LD + 7] += JT(-1.0 * dqdM);
      dwdC[5 * LD + 8] += JT(-1.0 * dqdM);
      PELEC_MEMORY_FENCE();
    }
    {  // R8: H + O2 (+M) <=> HO2 (+M)
      const double kinf = exp(28.019679105720332 + 0.6 * lnT);
      const double Mj = M1;
      const double k0r = exp(19.88299408302048 + -2.32 * lnT + -264.08961118015225 * invT);
      const double Pr = fmax(k0r * Mj, 1e-300);
      const double iPr1 = 1.0 / (1.0 + Pr);
      const double lFc = -0.09691001300805639;
      const double cc = -0.33507029128460225, nn = 0.8730757165202316;
      const double xx = log10(Pr) + cc;
      const double DD = 1.0 / (nn - 0.14 * xx);
      const double f1 = xx * DD;
      const double iden = 1.0 / (1.0 + f1 * f1);
      const double F = exp(-0.22314355131420974 * iden);
      const double g = -lFc * 2.0 * f1 * nn * DD * DD * iden * iden;
      const double dlnF_T = 0.0;
      const double kf = RMUL(kinf * Pr * iPr1 * F, 8);
      const double dlnkinf = (0.6 + 0.0 * invT) * invT;
      const double dlnPr = (-2.32 + 264.08961118015225 * invT) * invT;
      const double dkdM = RMUL(kinf * k0r * F * (iPr1 * iPr1 + g * iPr1), 8);
      const double dlnk = dlnkinf + dlnPr * iPr1 + g * dlnPr + dlnF_T;
      const double Pf = C[1] * C[3];
      const double iKc = (eg[6] * refC) / (eg[1] * eg[3]);
      const double Pb = C[6];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      const double dlnKc = (-1.0 * hRT[1] + -1.0 * hRT[3] + 1.0 * hRT[6] - -1.0) * invT;
      const double dqdT = kf * (dlnk * net + iKc * Pb * dlnKc);
      const double dq1 = kf * (C[3]);
      const double dq3 = kf * (C[1]);
      const double dq6 = -kf * iKc * (1.0);
      wd[1] += -1.0 * qj;
      dwdT[1] += -1.0 * dqdT;
      dwdC[1 * LD + 1] += JT(-1.0 * dq1);
      dwdC[1 * LD + 3] += JT(-1.0 * dq3);
      dwdC[1 * LD + 6] += JT(-1.0 * dq6);
      wd[3] += -1.0 * qj;
      dwdT[3] += -1.0 * dqdT;
      dwdC[3 * LD + 1] += JT(-1.0 * dq1);
      dwdC[3 * LD + 3] += JT(-1.0 * dq3);
      dwdC[3 * LD + 6] += JT(-1.0 * dq6);
      wd[6] += 1.0 * qj;
      dwdT[6] += 1.0 * dqdT;
      dwdC[6 * LD + 1] += JT(1.0 * dq1);
      dwdC[6 * LD + 3] += JT(1.0 * dq3);
      dwdC[6 * LD + 6] += JT(1.0 * dq6);
      const double dqdM = dkdM * net;
      dwdC[1 * LD + 0] += JT(-2.0 * dqdM);
      dwdC[1 * LD + 1] += JT(-0.78 * dqdM);
      dwdC[1 * LD + 2] += JT(-11.0 * dqdM);
      dwdC[1 * LD + 3] += JT(-1.0 * dqdM);
      dwdC[1 * LD + 4] += JT(-1.0 * dqdM);
      dwdC[1 * LD + 5] += JT(-1.0 * dqdM);
      dwdC[1 * LD + 6] += JT(-1.0 * dqdM);
      dwdC[1 * LD + 7] += JT(-1.0 * dqdM);
      dwdC[1 * LD + 8] += JT(-1.0 * dqdM);
      dwdC[3 * LD + 0] += JT(-2.0 * dqdM);
      dwdC[3 * LD + 1] += JT(-0.78 * dqdM);
      dwdC[3 * LD + 2] += JT(-11.0 * dqdM);
      dwdC[3 * LD + 3] += JT(-1.0 * dqdM);
      dwdC[3 * LD + 4] += JT(-1.0 * dqdM);
      dwdC[3 * LD + 5] += JT(-1.0 * dqdM);
      dwdC[3 * LD + 6] += JT(-1.0 * dqdM);
      dwdC[3 * LD + 7] += JT(-1.0 * dqdM);
      dwdC[3 * LD + 8] += JT(-1.0 * dqdM);
      dwdC[6 * LD + 0] += JT(2.0 * dqdM);
      dwdC[6 * LD + 1] += JT(0.78 * dqdM);
      dwdC[6 * LD + 2] += JT(11.0 * dqdM);
      dwdC[6 * LD + 3] += JT(1.0 * dqdM);
      dwdC[6 * LD + 4] += JT(1.0 * dqdM);
      dwdC[6 * LD + 5] += JT(1.0 * dqdM);
      dwdC[6 * LD + 6] += JT(1.0 * dqdM);
      dwdC[6 * LD + 7] += JT(1.0 * dqdM);
      dwdC[6 * LD + 8] += JT(1.0 * dqdM);
      PELEC_MEMORY_FENCE();
    }
    {  // R9: HO2 + H <=> H2 + O2
      const double kf = RMUL(exp(30.440423811291044 + -414.14967606948426 * invT), 9);
      const double dlnk = (0.0 + 414.14967606948426 * invT) * invT;
      const double Pf = C[3] * C[6];
      const double iKc = (eg[0] * eg[1]) / (eg[3] * eg[6]);
      const double Pb = C[0] * C[1];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      const double dlnKc = (1.0 * hRT[0] + 1.0 * hRT[1] + -1.0 * hRT[3] + -1.0 * hRT[6] - 0.0) * invT;
      const double dqdT = kf * (dlnk * net + iKc * Pb * dlnKc);
      const double dq0 = -kf * iKc * (C[1]);
      const double dq1 = -kf * iKc * (C[0]);
      const double dq3 = kf * (C[6]);
      const double dq6 = kf * (C[3]);
      wd[0] += 1.0 * qj;
      dwdT[0] += 1.0 * dqdT;
      dwdC[0 * LD + 0] += JT(1.0 * dq0);
      dwdC[0 * LD + 1] += JT(1.0 * dq1);
      dwdC[0 * LD + 3] += JT(1.0 * dq3);
      dwdC[0 * LD + 6] += JT(1.0 * dq6);
      wd[1] += 1.0 * qj;
      dwdT[1] += 1.0 * dqdT;
      dwdC[1 * LD + 0] += JT(1.0 * dq0);
      dwdC[1 * LD + 1] += JT(1.0 * dq1);
      dwdC[1 * LD + 3] += JT(1.0 * dq3);
      dwdC[1 * LD + 6] += JT(1.0 * dq6);
      wd[3] += -1.0 * qj;
      dwdT[3] += -1.0 * dqdT;
      dwdC[3 * LD + 0] += JT(-1.0 * dq0);
      dwdC[3 * LD + 1] += JT(-1.0 * dq1);
      dwdC[3 * LD + 3] += JT(-1.0 * dq3);
      dwdC[3 * LD + 6] += JT(-1.0 * dq6);
      wd[6] += -1.0 * qj;
      dwdT[6] += -1.0 * dqdT;
      dwdC[6 * LD + 0] += JT(-1.0 * dq0);
      dwdC[6 * LD + 1] += JT(-1.0 * dq1);
      dwdC[6 * LD + 3] += JT(-1.0 * dq3);
      dwdC[6 * LD + 6] += JT(-1.0 * dq6);
      PELEC_MEMORY_FENCE();
    }
    {  // R10: HO2 + H <=> OH + OH
      const double kf = RMUL(exp(31.890738863714645 + -148.4497623821359 * invT), 10);
      const double dlnk = (0.0 + 148.4497623821359 * invT) * invT;
      const double Pf = C[3] * C[6];
      const double iKc = (eg[5] * eg[5]) / (eg[3] * eg[6]);
      const double Pb = C[5] * C[5];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      const double dlnKc = (-1.0 * hRT[3] + 2.0 * hRT[5] + -1.0 * hRT[6] - 0.0) * invT;
      const double dqdT = kf * (dlnk * net + iKc * Pb * dlnKc);
      const double dq3 = kf * (C[6]);
      const double dq5 = -kf * iKc * (2.0 * C[5]);
      const double dq6 = kf * (C[3]);
      wd[3] += -1.0 * qj;
      dwdT[3] += -1.0 * dqdT;
      dwdC[3 * LD + 3] += JT(-1.0 * dq3);
      dwdC[3 * LD + 5] += JT(-1.0 * dq5);
      dwdC[3 * LD + 6] += JT(-1.0 * dq6);
      wd[5] += 2.0 * qj;
      dwdT[5] += 2.0 * dqdT;
      dwdC[5 * LD + 3] += JT(2.0 * dq3);
      dwdC[5 * LD + 5] += JT(2.0 * dq5);
      dwdC[5 * LD + 6] += JT(2.0 * dq6);
      wd[6] += -1.0 * qj;
      dwdT[6] += -1.0 * dqdT;
      dwdC[6 * LD + 3] += JT(-1.0 * dq3);
      dwdC[6 * LD + 5] += JT(-1.0 * dq5);
      dwdC[6 * LD + 6] += JT(-1.0 * dq6);
      PELEC_MEMORY_FENCE();
    }
    {  // R11: HO2 + O <=> O2 + OH
      const double kf = RMUL(32500000000000.0, 11);
      const double dlnk = (0.0 + 0.0 * invT) * invT;
      const double Pf = C[4] * C[6];
      const double iKc = (eg[1] * eg[5]) / (eg[4] * eg[6]);
      const double Pb = C[1] * C[5];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      const double dlnKc = (1.0 * hRT[1] + -1.0 * hRT[4] + 1.0 * hRT[5] + -1.0 * hRT[6] - 0.0) * invT;
      const double dqdT = kf * (dlnk * net + iKc * Pb * dlnKc);
      const double dq1 = -kf * iKc * (C[5]);
      const double dq4 = kf * (C[6]);
      const double dq5 = -kf * iKc * (C[1]);
      const double dq6 = kf * (C[4]);
      wd[1] += 1.0 * qj;
      dwdT[1] += 1.0 * dqdT;
      dwdC[1 * LD + 1] += JT(1.0 * dq1);
      dwdC[1 * LD + 4] += JT(1.0 * dq4);
      dwdC[1 * LD + 5] += JT(1.0 * dq5);
      dwdC[1 * LD + 6] += JT(1.0 * dq6);
      wd[4] += -1.0 * qj;
      dwdT[4] += -1.0 * dqdT;
      dwdC[4 * LD + 1] += JT(-1.0 * dq1);
      dwdC[4 * LD + 4] += JT(-1.0 * dq4);
      dwdC[4 * LD + 5] += JT(-1.0 * dq5);
      dwdC[4 * LD + 6] += JT(-1.0 * dq6);
      wd[5] += 1.0 * qj;
      dwdT[5] += 1.0 * dqdT;
      dwdC[5 * LD + 1] += JT(1.0 * dq1);
      dwdC[5 * LD + 4] += JT(1.0 * dq4);
      dwdC[5 * LD + 5] += JT(1.0 * dq5);
      dwdC[5 * LD + 6] += JT(1.0 * dq6);
      wd[6] += -1.0 * qj;
      dwdT[6] += -1.0 * dqdT;
      dwdC[6 * LD + 1] += JT(-1.0 * dq1);
      dwdC[6 * LD + 4] += JT(-1.0 * dq4);
      dwdC[6 * LD + 5] += JT(-1.0 * dq5);
      dwdC[6 * LD + 6] += JT(-1.0 * dq6);
      PELEC_MEMORY_FENCE();
    }
    {  // R12: HO2 + OH <=> H2O + O2
      const double kf = RMUL(exp(30.994862711046935 + 250.1001081488866 * invT), 12);
      const double dlnk = (0.0 + -250.1001081488866 * invT) * invT;
      const double Pf = C[5] * C[6];
      const double iKc = (eg[1] * eg[2]) / (eg[5] * eg[6]);
      const double Pb = C[1] * C[2];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      const double dlnKc = (1.0 * hRT[1] + 1.0 * hRT[2] + -1.0 * hRT[5] + -1.0 * hRT[6] - 0.0) * invT;
      const double dqdT = kf * (dlnk * net + iKc * Pb * dlnKc);
      const double dq1 = -kf * iKc * (C[2]);
      const double dq2 = -kf * iKc * (C[1]);
      const double dq5 = kf * (C[6]);
      const double dq6 = kf * (C[5]);
      wd[1] += 1.0 * qj;
      dwdT[1] += 1.0 * dqdT;
      dwdC[1 * LD + 1] += JT(1.0 * dq1);
      dwdC[1 * LD + 2] += JT(1.0 * dq2);
      dwdC[1 * LD + 5] += JT(1.0 * dq5);
      dwdC[1 * LD + 6] += JT(1.0 * dq6);
      wd[2] += 1.0 * qj;
      dwdT[2] += 1.0 * dqdT;
      dwdC[2 * LD + 1] += JT(1.0 * dq1);
      dwdC[2 * LD + 2] += JT(1.0 * dq2);
      dwdC[2 * LD + 5] += JT(1.0 * dq5);
      dwdC[2 * LD + 6] += JT(1.0 * dq6);
      wd[5] += -1.0 * qj;
      dwdT[5] += -1.0 * dqdT;
      dwdC[5 * LD + 1] += JT(-1.0 * dq1);
      dwdC[5 * LD + 2] += JT(-1.0 * dq2);
      dwdC[5 * LD + 5] += JT(-1.0 * dq5);
      dwdC[5 * LD + 6] += JT(-1.0 * dq6);
      wd[6] += -1.0 * qj;
      dwdT[6] += -1.0 * dqdT;
      dwdC[6 * LD + 1] += JT(-1.0 * dq1);
      dwdC[6 * LD + 2] += JT(-1.0 * dq2);
      dwdC[6 * LD + 5] += JT(-1.0 * dq5);
      dwdC[6 * LD + 6] += JT(-1.0 * dq6);
      PELEC_MEMORY_FENCE();
    }
    {  // R13: HO2 + HO2 <=> H2O2 + O2
      const double kf = RMUL(exp(33.67127582720596 + -6029.576450382212 * invT), 13);
      const double dlnk = (0.0 + 6029.576450382212 * invT) * invT;
      const double Pf = C[6] * C[6];
      const double iKc = (eg[1] * eg[7]) / (eg[6] * eg[6]);
      const double Pb = C[1] * C[7];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      const double dlnKc = (1.0 * hRT[1] + -2.0 * hRT[6] + 1.0 * hRT[7] - 0.0) * invT;
      const double dqdT = kf * (dlnk * net + iKc * Pb * dlnKc);
      const double dq1 = -kf * iKc * (C[7]);
      const double dq6 = kf * (2.0 * C[6]);
      const double dq7 = -kf * iKc * (C[1]);
      wd[1] += 1.0 * qj;
      dwdT[1] += 1.0 * dqdT;
      dwdC[1 * LD + 1] += JT(1.0 * dq1);
      dwdC[1 * LD + 6] += JT(1.0 * dq6);
      dwdC[1 * LD + 7] += JT(1.0 * dq7);
      wd[6] += -2.0 * qj;
      dwdT[6] += -2.0 * dqdT;
      dwdC[6 * LD + 1] += JT(-2.0 * dq1);
      dwdC[6 * LD + 6] += JT(-2.0 * dq6);
      dwdC[6 * LD + 7] += JT(-2.0 * dq7);
      wd[7] += 1.0 * qj;
      dwdT[7] += 1.0 * dqdT;
      dwdC[7 * LD + 1] += JT(1.0 * dq1);
      dwdC[7 * LD + 6] += JT(1.0 * dq6);
      dwdC[7 * LD + 7] += JT(1.0 * dq7);
      PELEC_MEMORY_FENCE();
    }
    {  // R14: HO2 + HO2 <=> H2O2 + O2
      const double kf = RMUL(exp(25.590800287401994 + 819.895585929539 * invT), 14);
      const double dlnk = (0.0 + -819.895585929539 * invT) * invT;
      const double Pf = C[6] * C[6];
      const double iKc = (eg[1] * eg[7]) / (eg[6] * eg[6]);
      const double Pb = C[1] * C[7];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      const double dlnKc = (1.0 * hRT[1] + -2.0 * hRT[6] + 1.0 * hRT[7] - 0.0) * invT;
      const double dqdT = kf * (dlnk * net + iKc * Pb * dlnKc);
      const double dq1 = -kf * iKc * (C[7]);
      const double dq6 = kf * (2.0 * C[6]);
      const double dq7 = -kf * iKc * (C[1]);
      wd[1] += 1.0 * qj;
      dwdT[1] += 1.0 * dqdT;
      dwdC[1 * LD + 1] += JT(1.0 * dq1);
      dwdC[1 * LD + 6] += JT(1.0 * dq6);
      dwdC[1 * LD + 7] += JT(1.0 * dq7);
      wd[6] += -2.0 * qj;
      dwdT[6] += -2.0 * dqdT;
      dwdC[6 * LD + 1] += JT(-2.0 * dq1);
      dwdC[6 * LD + 6] += JT(-2.0 * dq6);
      dwdC[6 * LD + 7] += JT(-2.0 * dq7);
      wd[7] += 1.0 * qj;
      dwdT[7] += 1.0 * dqdT;
      dwdC[7 * LD + 1] += JT(1.0 * dq1);
      dwdC[7 * LD + 6] += JT(1.0 * dq6);
      dwdC[7 * LD + 7] += JT(1.0 * dq7);
      PELEC_MEMORY_FENCE();
    }
    {  // R15: H2O2 (+M) <=> OH + OH (+M)
      const double kinf = exp(33.31833539787744 + -24370.922007345227 * invT);
      const double Mj = M0;
      const double k0r = exp(6.009598019134351 + 0.0 * lnT + 1474.4332331513833 * invT);
      const double Pr = fmax(k0r * Mj, 1e-300);
      const double iPr1 = 1.0 / (1.0 + Pr);
      const double lFc = -0.3010299956639812;
      const double cc = -0.19830990290513262, nn = 1.1323080944932562;
      const double xx = log10(Pr) + cc;
      const double DD = 1.0 / (nn - 0.14 * xx);
      const double f1 = xx * DD;
      const double iden = 1.0 / (1.0 + f1 * f1);
      const double F = exp(-0.6931471805599454 * iden);
      const double g = -lFc * 2.0 * f1 * nn * DD * DD * iden * iden;
      const double dlnF_T = 0.0;
      const double kf = RMUL(kinf * Pr * iPr1 * F, 15);
      const double dlnkinf = (0.0 + 24370.922007345227 * invT) * invT;
      const double dlnPr = (0.0 + -1474.4332331513833 * invT) * invT;
      const double dkdM = RMUL(kinf * k0r * F * (iPr1 * iPr1 + g * iPr1), 15);
      const double dlnk = dlnkinf + dlnPr * iPr1 + g * dlnPr + dlnF_T;
      const double Pf = C[7];
      const double iKc = (eg[5] * eg[5] * irefC) / (eg[7]);
      const double Pb = C[5] * C[5];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      const double dlnKc = (2.0 * hRT[5] + -1.0 * hRT[7] - 1.0) * invT;
      const double dqdT = kf * (dlnk * net + iKc * Pb * dlnKc);
      const double dq5 = -kf * iKc * (2.0 * C[5]);
      const double dq7 = kf * (1.0);
      wd[5] += 2.0 * qj;
      dwdT[5] += 2.0 * dqdT;
      dwdC[5 * LD + 5] += JT(2.0 * dq5);
      dwdC[5 * LD + 7] += JT(2.0 * dq7);
      wd[7] += -1.0 * qj;
      dwdT[7] += -1.0 * dqdT;
      dwdC[7 * LD + 5] += JT(-1.0 * dq5);
      dwdC[7 * LD + 7] += JT(-1.0 * dq7);
      const double dqdM = dkdM * net;
      dwdC[5 * LD + 0] += JT(5.0 * dqdM);
      dwdC[5 * LD + 1] += JT(2.0 * dqdM);
      dwdC[5 * LD + 2] += JT(24.0 * dqdM);
      dwdC[5 * LD + 3] += JT(2.0 * dqdM);
      dwdC[5 * LD + 4] += JT(2.0 * dqdM);
      dwdC[5 * LD + 5] += JT(2.0 * dqdM);
      dwdC[5 * LD + 6] += JT(2.0 * dqdM);
      dwdC[5 * LD + 7] += JT(2.0 * dqdM);
      dwdC[5 * LD + 8] += JT(2.0 * dqdM);
      dwdC[7 * LD + 0] += JT(-2.5 * dqdM);
      dwdC[7 * LD + 1] += JT(-1.0 * dqdM);
      dwdC[7 * LD + 2] += JT(-12.0 * dqdM);
      dwdC[7 * LD + 3] += JT(-1.0 * dqdM);
      dwdC[7 * LD + 4] += JT(-1.0 * dqdM);
      dwdC[7 * LD + 5] += JT(-1.0 * dqdM);
      dwdC[7 * LD + 6] += JT(-1.0 * dqdM);
      dwdC[7 * LD + 7] += JT(-1.0 * dqdM);
      dwdC[7 * LD + 8] += JT(-1.0 * dqdM);
      PELEC_MEMORY_FENCE();
    }
    {  // R16: H2O2 + H <=> H2O + OH
      const double kf = RMUL(exp(30.813232956425157 + -1997.7815479901 * invT), 16);
      const double dlnk = (0.0 + 1997.7815479901 * invT) * invT;
      const double Pf = C[3] * C[7];
      const double iKc = (eg[2] * eg[5]) / (eg[3] * eg[7]);
      const double Pb = C[2] * C[5];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      const double dlnKc = (1.0 * hRT[2] + -1.0 * hRT[3] + 1.0 * hRT[5] + -1.0 * hRT[7] - 0.0) * invT;
      const double dqdT = kf * (dlnk * net + iKc * Pb * dlnKc);
      const double dq2 = -kf * iKc * (C[5]);
      const double dq3 = kf * (C[7]);
      const double dq5 = -kf * iKc * (C[2]);
      const double dq7 = kf * (C[3]);
      wd[2] += 1.0 * qj;
      dwdT[2] += 1.0 * dqdT;
      dwdC[2 * LD + 2] += JT(1.0 * dq2);
      dwdC[2 * LD + 3] += JT(1.0 * dq3);
      dwdC[2 * LD + 5] += JT(1.0 * dq5);
      dwdC[2 * LD + 7] += JT(1.0 * dq7);
      wd[3] += -1.0 * qj;
      dwdT[3] += -1.0 * dqdT;
      dwdC[3 * LD + 2] += JT(-1.0 * dq2);
      dwdC[3 * LD + 3] += JT(-1.0 * dq3);
      dwdC[3 * LD + 5] += JT(-1.0 * dq5);
      dwdC[3 * LD + 7] += JT(-1.0 * dq7);
      wd[5] += 1.0 * qj;
      dwdT[5] += 1.0 * dqdT;
      dwdC[5 * LD + 2] += JT(1.0 * dq2);
      dwdC[5 * LD + 3] += JT(1.0 * dq3);
      dwdC[5 * LD + 5] += JT(1.0 * dq5);
      dwdC[5 * LD + 7] += JT(1.0 * dq7);
      wd[7] += -1.0 * qj;
      dwdT[7] += -1.0 * dqdT;
      dwdC[7 * LD + 2] += JT(-1.0 * dq2);
      dwdC[7 * LD + 3] += JT(-1.0 * dq3);
      dwdC[7 * LD + 5] += JT(-1.0 * dq5);
      dwdC[7 * LD + 7] += JT(-1.0 * dq7);
      PELEC_MEMORY_FENCE();
    }
    {  // R17: H2O2 + H <=> HO2 + H2
      const double kf = RMUL(exp(31.506380136985104 + -4000.595291315188 * invT), 17);
      const double dlnk = (0.0 + 4000.595291315188 * invT) * invT;
      const double Pf = C[3] * C[7];
      const double iKc = (eg[0] * eg[6]) / (eg[3] * eg[7]);
      const double Pb = C[0] * C[6];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      const double dlnKc = (1.0 * hRT[0] + -1.0 * hRT[3] + 1.0 * hRT[6] + -1.0 * hRT[7] - 0.0) * invT;
      const double dqdT = kf * (dlnk * net + iKc * Pb * dlnKc);
      const double dq0 = -kf * iKc * (C[6]);
      const double dq3 = kf * (C[7]);
      const double dq6 = -kf * iKc * (C[0]);
      const double dq7 = kf * (C[3]);
      wd[0] += 1.0 * qj;
      dwdT[0] += 1.0 * dqdT;
      dwdC[0 * LD + 0] += JT(1.0 * dq0);
      dwdC[0 * LD + 3] += JT(1.0 * dq3);
      dwdC[0 * LD + 6] += JT(1.0 * dq6);
      dwdC[0 * LD + 7] += JT(1.0 * dq7);
      wd[3] += -1.0 * qj;
      dwdT[3] += -1.0 * dqdT;
      dwdC[3 * LD + 0] += JT(-1.0 * dq0);
      dwdC[3 * LD + 3] += JT(-1.0 * dq3);
      dwdC[3 * LD + 6] += JT(-1.0 * dq6);
      dwdC[3 * LD + 7] += JT(-1.0 * dq7);
      wd[6] += 1.0 * qj;
      dwdT[6] += 1.0 * dqdT;
      dwdC[6 * LD + 0] += JT(1.0 * dq0);
      dwdC[6 * LD + 3] += JT(1.0 * dq3);
      dwdC[6 * LD + 6] += JT(1.0 * dq6);
      dwdC[6 * LD + 7] += JT(1.0 * dq7);
      wd[7] += -1.0 * qj;
      dwdT[7] += -1.0 * dqdT;
      dwdC[7 * LD + 0] += JT(-1.0 * dq0);
      dwdC[7 * LD + 3] += JT(-1.0 * dq3);
      dwdC[7 * LD + 6] += JT(-1.0 * dq6);
      dwdC[7 * LD + 7] += JT(-1.0 * dq7);
      PELEC_MEMORY_FENCE();
    }
    {  // R18: H2O2 + O <=> OH + HO2
      const double kf = RMUL(exp(16.07205171245691 + 2.0 * lnT + -1997.7815479901 * invT), 18);
      const double dlnk = (2.0 + 1997.7815479901 * invT) * invT;
      const double Pf = C[4] * C[7];
      const double iKc = (eg[5] * eg[6]) / (eg[4] * eg[7]);
      const double Pb = C[5] * C[6];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      const double dlnKc = (-1.0 * hRT[4] + 1.0 * hRT[5] + 1.0 * hRT[6] + -1.0 * hRT[7] - 0.0) * invT;
      const double dqdT = kf * (dlnk * net + iKc * Pb * dlnKc);
      const double dq4 = kf * (C[7]);
      const double dq5 = -kf * iKc * (C[6]);
      const double dq6 = -kf * iKc * (C[5]);
      const double dq7 = kf * (C[4]);
      wd[4] += -1.0 * qj;
      dwdT[4] += -1.0 * dqdT;
      dwdC[4 * LD + 4] += JT(-1.0 * dq4);
      dwdC[4 * LD + 5] += JT(-1.0 * dq5);
      dwdC[4 * LD + 6] += JT(-1.0 * dq6);
      dwdC[4 * LD + 7] += JT(-1.0 * dq7);
      wd[5] += 1.0 * qj;
      dwdT[5] += 1.0 * dqdT;
      dwdC[5 * LD + 4] += JT(1.0 * dq4);
      dwdC[5 * LD + 5] += JT(1.0 * dq5);
      dwdC[5 * LD + 6] += JT(1.0 * dq6);
      dwdC[5 * LD + 7] += JT(1.0 * dq7);
      wd[6] += 1.0 * qj;
      dwdT[6] += 1.0 * dqdT;
      dwdC[6 * LD + 4] += JT(1.0 * dq4);
      dwdC[6 * LD + 5] += JT(1.0 * dq5);
      dwdC[6 * LD + 6] += JT(1.0 * dq6);
      dwdC[6 * LD + 7] += JT(1.0 * dq7);
      wd[7] += -1.0 * qj;
      dwdT[7] += -1.0 * dqdT;
      dwdC[7 * LD + 4] += JT(-1.0 * dq4);
      dwdC[7 * LD + 5] += JT(-1.0 * dq5);
      dwdC[7 * LD + 6] += JT(-1.0 * dq6);
      dwdC[7 * LD + 7] += JT(-1.0 * dq7);
      PELEC_MEMORY_FENCE();
    }
    {  // R19: H2O2 + OH <=> HO2 + H2O
      const double kf = RMUL(1000000000000.0, 19);
      const double dlnk = (0.0 + 0.0 * invT) * invT;
      const double Pf = C[5] * C[7];
      const double iKc = (eg[2] * eg[6]) / (eg[5] * eg[7]);
      const double Pb = C[2] * C[6];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      const double dlnKc = (1.0 * hRT[2] + -1.0 * hRT[5] + 1.0 * hRT[6] + -1.0 * hRT[7] - 0.0) * invT;
      const double dqdT = kf * (dlnk * net + iKc * Pb * dlnKc);
      const double dq2 = -kf * iKc * (C[6]);
      const double dq5 = kf * (C[7]);
      const double dq6 = -kf * iKc * (C[2]);
      const double dq7 = kf * (C[5]);
      wd[2] += 1.0 * qj;
      dwdT[2] += 1.0 * dqdT;
      dwdC[2 * LD + 2] += JT(1.0 * dq2);
      dwdC[2 * LD + 5] += JT(1.0 * dq5);
      dwdC[2 * LD + 6] += JT(1.0 * dq6);
      dwdC[2 * LD + 7] += JT(1.0 * dq7);
      wd[5] += -1.0 * qj;
      dwdT[5] += -1.0 * dqdT;
      dwdC[5 * LD + 2] += JT(-1.0 * dq2);
      dwdC[5 * LD + 5] += JT(-1.0 * dq5);
      dwdC[5 * LD + 6] += JT(-1.0 * dq6);
      dwdC[5 * LD + 7] += JT(-1.0 * dq7);
      wd[6] += 1.0 * qj;
      dwdT[6] += 1.0 * dqdT;
      dwdC[6 * LD + 2] += JT(1.0 * dq2);
      dwdC[6 * LD + 5] += JT(1.0 * dq5);
      dwdC[6 * LD + 6] += JT(1.0 * dq6);
      dwdC[6 * LD + 7] += JT(1.0 * dq7);
      wd[7] += -1.0 * qj;
      dwdT[7] += -1.0 * dqdT;
      dwdC[7 * LD + 2] += JT(-1.0 * dq2);
      dwdC[7 * LD + 5] += JT(-1.0 * dq5);
      dwdC[7 * LD + 6] += JT(-1.0 * dq6);
      dwdC[7 * LD + 7] += JT(-1.0 * dq7);
      PELEC_MEMORY_FENCE();
    }
    {  // R20: H2O2 + OH <=> HO2 + H2O
      const double kf = RMUL(exp(33.99404921946901 + -4809.269081647704 * invT), 20);
      const double dlnk = (0.0 + 4809.269081647704 * invT) * invT;
      const double Pf = C[5] * C[7];
      const double iKc = (eg[2] * eg[6]) / (eg[5] * eg[7]);
      const double Pb = C[2] * C[6];
      const double net = Pf - iKc * Pb;
      const double qj = kf * net;
      const double dlnKc = (1.0 * hRT[2] + -1.0 * hRT[5] + 1.0 * hRT[6] + -1.0 * hRT[7] - 0.0) * invT;
      const double dqdT = kf * (dlnk * net + iKc * Pb * dlnKc);
      const double dq2 = -kf * iKc * (C[6]);
      const double dq5 = kf * (C[7]);
      const double dq6 = -kf * iKc * (C[2]);
      const double dq7 = kf * (C[5]);
      wd[2] += 1.0 * qj;
      dwdT[2] += 1.0 * dqdT;
      dwdC[2 * LD + 2] += JT(1.0 * dq2);
      dwdC[2 * LD + 5] += JT(1.0 * dq5);
      dwdC[2 * LD + 6] += JT(1.0 * dq6);
      dwdC[2 * LD + 7] += JT(1.0 * dq7);
      wd[5] += -1.0 * qj;
      dwdT[5] += -1.0 * dqdT;
      dwdC[5 * LD + 2] += JT(-1.0 * dq2);
      dwdC[5 * LD + 5] += JT(-1.0 * dq5);
      dwdC[5 * LD + 6] += JT(-1.0 * dq6);
      dwdC[5 * LD + 7] += JT(-1.0 * dq7);
      wd[6] += 1.0 * qj;
      dwdT[6] += 1.0 * dqdT;
      dwdC[6 * LD + 2] += JT(1.0 * dq2);
      dwdC[6 * LD + 5] += JT(1.0 * dq5);
      dwdC[6 * LD + 6] += JT(1.0 * dq6);
      dwdC[6 * LD + 7] += JT(1.0 * dq7);
      wd[7] += -1.0 * qj;
      dwdT[7] += -1.0 * dqdT;
      dwdC[7 * LD + 2] += JT(-1.0 * dq2);
      dwdC[7 * LD + 5] += JT(-1.0 * dq5);
      dwdC[7 * LD + 6] += JT(-1.0 * dq6);
      dwdC[7 * LD + 7] += JT(-1.0 * dq7);
      PELEC_MEMORY_FENCE();
    }
    {  // R21: 2 H + 2 OH => 2 H2O
      const double kf = RMUL(1e+27, 21);
      const double dlnk = (0.0 + 0.0 * invT) * invT;
      const double Pf = C[3] * C[3] * C[5] * C[5];
      const double net = Pf;
      const double qj = kf * net;
      const double dqdT = kf * dlnk * net;
      const double dq3 = kf * (2.0 * C[3] * C[5] * C[5]);
      const double dq5 = kf * (2.0 * C[5] * C[3] * C[3]);
      wd[2] += 2.0 * qj;
      dwdT[2] += 2.0 * dqdT;
      dwdC[2 * LD + 3] += JT(2.0 * dq3);
      dwdC[2 * LD + 5] += JT(2.0 * dq5);
      wd[3] += -2.0 * qj;
      dwdT[3] += -2.0 * dqdT;
      dwdC[3 * LD + 3] += JT(-2.0 * dq3);
      dwdC[3 * LD + 5] += JT(-2.0 * dq5);
      wd[5] += -2.0 * qj;
      dwdT[5] += -2.0 * dqdT;
      dwdC[5 * LD + 3] += JT(-2.0 * dq3);
      dwdC[5 * LD + 5] += JT(-2.0 * dq5);
      PELEC_MEMORY_FENCE();
    }
  }
  // out[j] = sum_k nu_kj w[k] (net stoichiometric coefficients, products minus reactants)
  __host__ __device__ static inline void nu_dot(const double* w, double* out) {
    out[0] = -1.0 * w[1] + -1.0 * w[3] + 1.0 * w[4] + 1.0 * w[5];
    out[1] = -1.0 * w[0] + 1.0 * w[3] + -1.0 * w[4] + 1.0 * w[5];
    out[2] = -1.0 * w[0] + 1.0 * w[2] + 1.0 * w[3] + -1.0 * w[5];
    out[3] = -1.0 * w[2] + -1.0 * w[4] + 2.0 * w[5];
    out[4] = -1.0 * w[0] + 2.0 * w[3];
    out[5] = 1.0 * w[1] + -2.0 * w[4];
    out[6] = -1.0 * w[3] + -1.0 * w[4] + 1.0 * w[5];
    out[7] = 1.0 * w[2] + -1.0 * w[3] + -1.0 * w[5];
    out[8] = -1.0 * w[1] + -1.0 * w[3] + 1.0 * w[6];
    out[9] = 1.0 * w[0] + 1.0 * w[1] + -1.0 * w[3] + -1.0 * w[6];
    out[10] = -1.0 * w[3] + 2.0 * w[5] + -1.0 * w[6];
    out[11] = 1.0 * w[1] + -1.0 * w[4] + 1.0 * w[5] + -1.0 * w[6];
    out[12] = 1.0 * w[1] + 1.0 * w[2] + -1.0 * w[5] + -1.0 * w[6];
    out[13] = 1.0 * w[1] + -2.0 * w[6] + 1.0 * w[7];
    out[14] = 1.0 * w[1] + -2.0 * w[6] + 1.0 * w[7];
    out[15] = 2.0 * w[5] + -1.0 * w[7];
    out[16] = 1.0 * w[2] + -1.0 * w[3] + 1.0 * w[5] + -1.0 * w[7];
    out[17] = 1.0 * w[0] + -1.0 * w[3] + 1.0 * w[6] + -1.0 * w[7];
    out[18] = -1.0 * w[4] + 1.0 * w[5] + 1.0 * w[6] + -1.0 * w[7];
    out[19] = 1.0 * w[2] + -1.0 * w[5] + 1.0 * w[6] + -1.0 * w[7];
    out[20] = 1.0 * w[2] + -1.0 * w[5] + 1.0 * w[6] + -1.0 * w[7];
    out[21] = 2.0 * w[2] + -2.0 * w[3] + -2.0 * w[5];
  }
  static constexpr bool T_OK = true;
  // ---- data tables (cooperative kernels)
  static constexpr double T_REFC = 0.012186596374704216;  // P_atm / R, times 1/T
  static constexpr double T_IREFC = 82.05736608095968;
  static constexpr double T_LN10 = 2.302585092994046;
  static constexpr double T_TMID[9] = {1000.0, 1000.0, 1000.0, 1000.0, 1000.0, 1000.0, 1000.0, 1000.0, 1000.0};
  static constexpr int T_TMIDG[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  static constexpr double T_G[9][2][7] = {{{6.592218, -0.0004124721, 1.3571691666666666e-07, 7.896194999999999e-12, -2.067436e-14, 3.298124, -1012.521}, {4.346533, -0.0003500322, 9.389715e-09, 7.692981666666667e-13, -7.91376e-17, 2.991423, -835.034}}, {{-2.821802, -0.000563743, 9.593583333333333e-08, -1.0948975000000001e-10, 4.384277e-14, 3.212936, -1005.249}, {0.5084119999999999, -0.00030675985, 2.09807e-08, -1.4794008333333333e-12, 5.682175000000001e-17, 3.697578, -1233.93}}, {{0.7966090000000001, -0.001737491, 1.059116e-06, -5.807150833333333e-10, 1.2532940000000001e-13, 3.386842, -30208.11}, {-4.190671, -0.0015281465, 1.4550433333333335e-07, -1.00083e-11, 3.195809e-16, 2.672146, -29899.21}}, {{2.9601176000000002, 0.0, 0.0, 0.0, 0.0, 2.5, 25471.63}, {2.9601176000000002, 0.0, 0.0, 0.0, 0.0, 2.5, 25471.63}}, {{-0.01756599999999997, 0.000819083, -4.035053333333333e-07, 1.3357024999999999e-10, -1.945348e-14, 2.946429, 29147.64}, {-2.378248, 1.377531e-05, 5.171338333333333e-10, -3.7925558333333335e-13, 2.184026e-17, 2.54206, 29230.8}}, {{4.81573857, 0.001612724695, -1.0879411516666667e-06, 4.832113691666666e-10, -1.0311868949999999e-13, 4.12530561, 3346.30913}, {-2.8369118700000002, -0.00052825224, 4.318045966666667e-08, -2.54348895e-12, 6.6597938e-17, 2.86472886, 3683.62875}}, {{0.5851355599999999, 0.002374560255, -3.5263815166666663e-06, 2.02303245e-09, -4.646125620000001e-13, 4.30179801, 294.80804}, {0.23210875000000009, -0.001119910065, 1.0560969166666666e-07, -9.520530833333334e-12, 5.39542675e-16, 4.0172109, 111.856713}}, {{-3.396609, -0.003284613, 2.4750216666666664e-08, 3.854838333333333e-10, -1.2357574999999998e-13, 3.388754, -17663.15}, {4.07203, -0.002168068, 2.457815e-07, -1.9574199999999998e-11, 7.15827e-16, 4.573167, -18006.96}}, {{-0.6516950000000001, -0.00070412, 6.605369999999999e-07, -4.701262500000001e-10, 1.2224275000000001e-13, 3.298677, -1020.9}, {-3.0538879999999997, -0.0007439885, 9.474601666666666e-08, -8.4142e-12, 3.3766754999999997e-16, 2.92664, -922.7977}}};
  static constexpr double T_H[9][2][6] = {{{3.298124, 0.0004124721, -2.714338333333333e-07, -2.3688585e-11, 8.269744e-14, -1012.521}, {2.991423, 0.0003500322, -1.877943e-08, -2.3078945e-12, 3.165504e-16, -835.034}}, {{3.212936, 0.000563743, -1.9187166666666667e-07, 3.2846925e-10, -1.7537108e-13, -1005.249}, {3.697578, 0.00030675985, -4.19614e-08, 4.4382025e-12, -2.2728700000000004e-16, -1233.93}}, {{3.386842, 0.001737491, -2.118232e-06, 1.74214525e-09, -5.013176000000001e-13, -30208.11}, {2.672146, 0.0015281465, -2.910086666666667e-07, 3.00249e-11, -1.2783236e-15, -29899.21}}, {{2.5, 0.0, 0.0, 0.0, 0.0, 25471.63}, {2.5, 0.0, 0.0, 0.0, 0.0, 25471.63}}, {{2.946429, -0.000819083, 8.070106666666666e-07, -4.0071075e-10, 7.781392e-14, 29147.64}, {2.54206, -1.377531e-05, -1.0342676666666666e-09, 1.13776675e-12, -8.736104e-17, 29230.8}}, {{4.12530561, -0.001612724695, 2.1758823033333334e-06, -1.4496341075e-09, 4.1247475799999997e-13, 3346.30913}, {2.86472886, 0.00052825224, -8.636091933333334e-08, 7.63046685e-12, -2.66391752e-16, 3683.62875}}, {{4.30179801, -0.002374560255, 7.0527630333333326e-06, -6.06909735e-09, 1.8584502480000002e-12, 294.80804}, {4.0172109, 0.001119910065, -2.1121938333333332e-07, 2.85615925e-11, -2.1581707e-15, 111.856713}}, {{3.388754, 0.003284613, -4.950043333333333e-08, -1.1564515e-09, 4.943029999999999e-13, -17663.15}, {4.573167, 0.002168068, -4.91563e-07, 5.87226e-11, -2.863308e-15, -18006.96}}, {{3.298677, 0.00070412, -1.3210739999999999e-06, 1.41037875e-09, -4.889710000000001e-13, -1020.9}, {2.92664, 0.0007439885, -1.8949203333333333e-07, 2.52426e-11, -1.3506701999999999e-15, -922.7977}}};
  static constexpr double T_E[9][2][6] = {{{-41760012721.584656, 94782910.65151145, 17011.834957792224, -11.194908878994598, -0.0009770025618790518, 3.4107402675524593e-06}, {-34439809606.868126, 82133456.80144538, 14436.58859911475, -0.7745313289345194, -9.518588126080866e-05, 1.3055678579528436e-08}}, {{-2612005835.355053, 5750019.890860144, 1464.8112115909228, -0.498553008232421, 0.0008534836619928971, -4.5567842824267206e-07}, {-3206203000.868104, 7009297.673835451, 797.0746732925282, -0.1090311173248295, 1.153207894609931e-05, -5.905750419053826e-10}}, {{-139416853281.73718, 11015783.540270746, 8018.89055042963, -9.776091253662699, 0.00804037090419511, -2.3136873603397435e-06}, {-137991214074.95697, 7717309.475754812, 7052.721152812942, -1.343066897743044, 0.00013857130016074593, -5.899735328949149e-09}}, {{2101083518938.3674, 123730804.75837436, 0.0, 0.0, 0.0, 0.0}, {2101083518938.3674, 123730804.75837436, 0.0, 0.0, 0.0, 0.0}}, {{151472532212.07553, 10115073.789885493, -4256.556486283742, 4.193819781023616, -0.0020823871842488772, 4.043782448166599e-07}, {151904692612.66907, 8013675.653430371, -71.58662202862139, -0.005374813962813966, 5.912671169576799e-06, -4.5399208805517084e-10}}, {{16359238477.301249, 15278809.51884366, -7884.193258540319, 10.637324920058875, -0.0070868856247666085, 2.0164822405361935e-06}, {18008306717.04652, 9116176.33970538, 2582.488357950532, -0.42219616287900336, 3.7303375762027e-05, -1.302320266912726e-09}}, {{742626566.6440628, 8317286.461788826, -5981.558472625442, 17.766032421634424, -0.015288161502173006, 4.681468412296513e-06}, {281769000.368105, 7600406.5951120015, 2821.072880241255, -0.5320652905311182, 7.194714695081523e-05, -5.436469429981671e-09}}, {{-43175282361.06859, 5838999.75039175, 8028.811040037399, -0.12099739775532213, -0.0028267959027342975, 1.2082596590598668e-06}, {-44015681374.1868, 8734143.91817158, 5299.561407676278, -1.2015620839575023, 0.0001435397896737607, -6.998985536934612e-09}}, {{-3030062358.3258877, 6822543.492653029, 2089.8496500582078, -3.9209879517709996, 0.004186047175392025, -1.4512808516142303e-06}, {-2738891737.799691, 5718326.321916925, 2208.180574862709, -0.5624181383151804, 7.492080721547366e-05, -4.0088303766602985e-09}}};
  static constexpr double T_CV[9][2][5] = {{{94782910.65151145, 34023.66991558445, -33.584726636983795, -0.003908010247516207, 1.7053701337762297e-05}, {82133456.80144538, 28873.1771982295, -2.323593986803558, -0.00038074352504323465, 6.527839289764218e-08}}, {{5750019.890860144, 2929.6224231818455, -1.495659024697263, 0.0034139346479715883, -2.2783921412133602e-06}, {7009297.673835451, 1594.1493465850565, -0.32709335197448847, 4.612831578439724e-05, -2.952875209526913e-09}}, {{11015783.540270746, 16037.78110085926, -29.328273760988097, 0.03216148361678044, -1.1568436801698717e-05}, {7717309.475754812, 14105.442305625884, -4.029200693229132, 0.0005542852006429837, -2.9498676644745744e-08}}, {{123730804.75837436, 0.0, 0.0, 0.0, 0.0}, {123730804.75837436, 0.0, 0.0, 0.0, 0.0}}, {{10115073.789885493, -8513.112972567484, 12.581459343070849, -0.008329548736995509, 2.0218912240832993e-06}, {8013675.653430371, -143.17324405724278, -0.016124441888441896, 2.3650684678307196e-05, -2.269960440275854e-09}}, {{15278809.51884366, -15768.386517080638, 31.911974760176626, -0.028347542499066434, 1.0082411202680968e-05}, {9116176.33970538, 5164.976715901064, -1.26658848863701, 0.000149213503048108, -6.51160133456363e-09}}, {{8317286.461788826, -11963.116945250884, 53.29809726490328, -0.061152646008692024, 2.3407342061482568e-05}, {7600406.5951120015, 5642.14576048251, -1.5961958715933544, 0.0002877885878032609, -2.7182347149908354e-08}}, {{5838999.75039175, 16057.622080074798, -0.3629921932659664, -0.01130718361093719, 6.041298295299334e-06}, {8734143.91817158, 10599.122815352555, -3.604686251872507, 0.0005741591586950428, -3.499492768467306e-08}}, {{6822543.492653029, 4179.6993001164155, -11.762963855312998, 0.0167441887015681, -7.256404258071151e-06}, {5718326.321916925, 4416.361149725418, -1.6872544149455413, 0.00029968322886189463, -2.004415188330149e-08}}};
  static constexpr double T_DCV[9][2][4] = {{{34023.66991558445, -67.16945327396759, -0.011724030742548621, 6.821480535104919e-05}, {28873.1771982295, -4.647187973607116, -0.001142230575129704, 2.611135715905687e-07}}, {{2929.6224231818455, -2.991318049394526, 0.010241803943914765, -9.113568564853441e-06}, {1594.1493465850565, -0.6541867039489769, 0.0001383849473531917, -1.1811500838107651e-08}}, {{16037.78110085926, -58.656547521976194, 0.09648445085034131, -4.627374720679487e-05}, {14105.442305625884, -8.058401386458264, 0.001662855601928951, -1.1799470657898298e-07}}, {{0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}}, {{-8513.112972567484, 25.162918686141698, -0.024988646210986527, 8.087564896333197e-06}, {-143.17324405724278, -0.03224888377688379, 7.095205403492159e-05, -9.079841761103417e-09}}, {{-15768.386517080638, 63.82394952035325, -0.0850426274971993, 4.032964481072387e-05}, {5164.976715901064, -2.53317697727402, 0.00044764050914432405, -2.604640533825452e-08}}, {{-11963.116945250884, 106.59619452980655, -0.18345793802607607, 9.362936824593027e-05}, {5642.14576048251, -3.192391743186709, 0.0008633657634097827, -1.0872938859963342e-07}}, {{16057.622080074798, -0.7259843865319328, -0.03392155083281157, 2.4165193181197337e-05}, {10599.122815352555, -7.209372503745014, 0.0017224774760851284, -1.3997971073869224e-07}}, {{4179.6993001164155, -23.525927710625997, 0.05023256610470429, -2.9025617032284605e-05}, {4416.361149725418, -3.3745088298910826, 0.0008990496865856839, -8.017660753320596e-08}}};
  static constexpr int T_NSETS = 2;
  static constexpr double T_EFFD[2][9] = {{1.5, 0.0, 11.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, {1.0, -0.21999999999999997, 10.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0}};
  static constexpr double T_EFFV[2][9] = {{2.5, 1.0, 12.0, 1.0, 1.0, 1.0, 1.0, 1.0, 1.0}, {2.0, 0.78, 11.0, 1.0, 1.0, 1.0, 1.0, 1.0, 1.0}};
  static constexpr int T_RORD[22] = {8, 15, 4, 5, 6, 7, 0, 1, 2, 3, 9, 10, 11, 12, 13, 14, 16, 17, 18, 19, 20, 21};
  static constexpr int T_KIND[22] = {0, 0, 0, 0, 1, 1, 1, 1, 2, 0, 0, 0, 0, 0, 0, 2, 0, 0, 0, 0, 0, 0};
  static constexpr int T_REV[22] = {1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 0};
  static constexpr int T_KCONST[22] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 1, 0, 0, 0, 0, 0, 0, 0, 1, 0, 1};
  static constexpr double T_A[22] = {3547000000000000.0, 50800.0, 216000000.0, 2970000.0, 4.577e+19, 6165000000000000.0, 4.714e+18, 3.8e+22, 1475000000000.0, 16600000000000.0, 70790000000000.0, 32500000000000.0, 28900000000000.0, 420000000000000.0, 130000000000.0, 295100000000000.0, 24100000000000.0, 48200000000000.0, 9550000.0, 1000000000000.0, 580000000000000.0, 1e+27};
  static constexpr double T_LNA[22] = {35.80487857070217, 10.835651633566574, 19.19078896564844, 14.904072510778882, 45.27016052855837, 36.35766453152699, 42.99706847840676, 51.99187311260135, 28.019679105720332, 30.440423811291044, 31.890738863714645, 31.11226120526424, 30.994862711046935, 33.67127582720596, 25.590800287401994, 33.31833539787744, 30.813232956425157, 31.506380136985104, 16.07205171245691, 27.631021115928547, 33.99404921946901, 62.16979751083923};
  static constexpr double T_B[22] = {-0.406, 2.67, 1.51, 2.02, -1.4, -0.5, -1.0, -2.0, 0.6, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 2.0, 0.0, 0.0, 0.0};
  static constexpr double T_EAR[22] = {8352.941036546013, 3165.2508657072367, 1726.0429999007667, 6743.141748883461, 52526.05490660117, 0.0, 0.0, 0.0, 0.0, 414.14967606948426, 148.4497623821359, 0.0, -250.1001081488866, 6029.576450382212, -819.895585929539, 24370.922007345227, 1997.7815479901, 4000.595291315188, 1997.7815479901, 0.0, 4809.269081647704, 0.0};
  static constexpr double T_LOW[22][3] = {{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, {19.88299408302048, -2.32, 264.08961118015225}, {0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, {6.009598019134351, 0.0, -1474.4332331513833}, {0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}};
  static constexpr int T_TROEK[22] = {0, 0, 0, 0, 0, 0, 0, 0, 1, 0, 0, 0, 0, 0, 0, 1, 0, 0, 0, 0, 0, 0};
  static constexpr double T_TROE[22][8] = {{0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, {-0.09691001300805639, -0.33507029128460225, 0.8730757165202316, -0.22314355131420974, 0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, {-0.3010299956639812, -0.19830990290513262, 1.1323080944932562, -0.6931471805599454, 0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0}};
  static constexpr int T_EFF[22] = {-1, -1, -1, -1, 0, 0, 0, 0, 1, -1, -1, -1, -1, -1, -1, 0, -1, -1, -1, -1, -1, -1};
  static constexpr int T_RSP[22][3] = {{1, 3, -1}, {0, 4, -1}, {0, 5, -1}, {2, 4, -1}, {0, -1, -1}, {4, -1, -1}, {3, 4, -1}, {3, 5, -1}, {1, 3, -1}, {3, 6, -1}, {3, 6, -1}, {4, 6, -1}, {5, 6, -1}, {6, -1, -1}, {6, -1, -1}, {7, -1, -1}, {3, 7, -1}, {3, 7, -1}, {4, 7, -1}, {5, 7, -1}, {5, 7, -1}, {3, 5, -1}};
  static constexpr int T_RNU[22][3] = {{1, 1, 0}, {1, 1, 0}, {1, 1, 0}, {1, 1, 0}, {1, 0, 0}, {2, 0, 0}, {1, 1, 0}, {1, 1, 0}, {1, 1, 0}, {1, 1, 0}, {1, 1, 0}, {1, 1, 0}, {1, 1, 0}, {2, 0, 0}, {2, 0, 0}, {1, 0, 0}, {1, 1, 0}, {1, 1, 0}, {1, 1, 0}, {1, 1, 0}, {1, 1, 0}, {2, 2, 0}};
  static constexpr int T_PSP[22][3] = {{4, 5, -1}, {3, 5, -1}, {2, 3, -1}, {5, -1, -1}, {3, -1, -1}, {1, -1, -1}, {5, -1, -1}, {2, -1, -1}, {6, -1, -1}, {0, 1, -1}, {5, -1, -1}, {1, 5, -1}, {1, 2, -1}, {1, 7, -1}, {1, 7, -1}, {5, -1, -1}, {2, 5, -1}, {0, 6, -1}, {5, 6, -1}, {2, 6, -1}, {2, 6, -1}, {-1, -1, -1}};
  static constexpr int T_PNU[22][3] = {{1, 1, 0}, {1, 1, 0}, {1, 1, 0}, {2, 0, 0}, {2, 0, 0}, {1, 0, 0}, {1, 0, 0}, {1, 0, 0}, {1, 0, 0}, {1, 1, 0}, {2, 0, 0}, {1, 1, 0}, {1, 1, 0}, {1, 1, 0}, {1, 1, 0}, {2, 0, 0}, {1, 1, 0}, {1, 1, 0}, {1, 1, 0}, {1, 1, 0}, {1, 1, 0}, {0, 0, 0}};
  static constexpr int T_DNU[22] = {0, 0, 0, 0, 1, -1, -1, -1, -1, 0, 0, 0, 0, 0, 0, 1, 0, 0, 0, 0, 0, 0};
  static constexpr int T_NSPC[22][6] = {{1, 3, 4, 5, -1, -1}, {0, 3, 4, 5, -1, -1}, {0, 2, 3, 5, -1, -1}, {2, 4, 5, -1, -1, -1}, {0, 3, -1, -1, -1, -1}, {1, 4, -1, -1, -1, -1}, {3, 4, 5, -1, -1, -1}, {2, 3, 5, -1, -1, -1}, {1, 3, 6, -1, -1, -1}, {0, 1, 3, 6, -1, -1}, {3, 5, 6, -1, -1, -1}, {1, 4, 5, 6, -1, -1}, {1, 2, 5, 6, -1, -1}, {1, 6, 7, -1, -1, -1}, {1, 6, 7, -1, -1, -1}, {5, 7, -1, -1, -1, -1}, {2, 3, 5, 7, -1, -1}, {0, 3, 6, 7, -1, -1}, {4, 5, 6, 7, -1, -1}, {2, 5, 6, 7, -1, -1}, {2, 5, 6, 7, -1, -1}, {2, 3, 5, -1, -1, -1}};
  static constexpr double T_NNU[22][6] = {{-1.0, -1.0, 1.0, 1.0, 0.0, 0.0}, {-1.0, 1.0, -1.0, 1.0, 0.0, 0.0}, {-1.0, 1.0, 1.0, -1.0, 0.0, 0.0}, {-1.0, -1.0, 2.0, 0.0, 0.0, 0.0}, {-1.0, 2.0, 0.0, 0.0, 0.0, 0.0}, {1.0, -2.0, 0.0, 0.0, 0.0, 0.0}, {-1.0, -1.0, 1.0, 0.0, 0.0, 0.0}, {1.0, -1.0, -1.0, 0.0, 0.0, 0.0}, {-1.0, -1.0, 1.0, 0.0, 0.0, 0.0}, {1.0, 1.0, -1.0, -1.0, 0.0, 0.0}, {-1.0, 2.0, -1.0, 0.0, 0.0, 0.0}, {1.0, -1.0, 1.0, -1.0, 0.0, 0.0}, {1.0, 1.0, -1.0, -1.0, 0.0, 0.0}, {1.0, -2.0, 1.0, 0.0, 0.0, 0.0}, {1.0, -2.0, 1.0, 0.0, 0.0, 0.0}, {2.0, -1.0, 0.0, 0.0, 0.0, 0.0}, {1.0, -1.0, 1.0, -1.0, 0.0, 0.0}, {1.0, -1.0, 1.0, -1.0, 0.0, 0.0}, {-1.0, 1.0, 1.0, -1.0, 0.0, 0.0}, {1.0, -1.0, 1.0, -1.0, 0.0, 0.0}, {1.0, -1.0, 1.0, -1.0, 0.0, 0.0}, {2.0, -2.0, -2.0, 0.0, 0.0, 0.0}};
  static constexpr int T_CSR_MAX = 15;
  static constexpr int T_CSR_PTR[10] = {0, 5, 13, 21, 33, 40, 55, 66, 74, 74};
  static constexpr int T_CSR_PAD = 8;
  static constexpr int T_CSR_J[82] = {1, 2, 4, 9, 17, 0, 5, 8, 9, 11, 12, 13, 14, 2, 3, 7, 12, 16, 19, 20, 21, 0, 1, 2, 4, 6, 7, 8, 9, 10, 16, 17, 21, 0, 1, 3, 5, 6, 11, 18, 0, 1, 2, 3, 6, 7, 10, 11, 12, 15, 16, 18, 19, 20, 21, 8, 9, 10, 11, 12, 13, 14, 17, 18, 19, 20, 13, 14, 15, 16, 17, 18, 19, 20, 0, 0, 0, 0, 0, 0, 0, 0};
  static constexpr double T_CSR_NU[82] = {-1.0, -1.0, -1.0, 1.0, 1.0, -1.0, 1.0, -1.0, 1.0, 1.0, 1.0, 1.0, 1.0, 1.0, -1.0, 1.0, 1.0, 1.0, 1.0, 1.0, 2.0, -1.0, 1.0, 1.0, 2.0, -1.0, -1.0, -1.0, -1.0, -1.0, -1.0, -1.0, -2.0, 1.0, -1.0, -1.0, -2.0, -1.0, -1.0, -1.0, 1.0, 1.0, -1.0, 2.0, 1.0, -1.0, 2.0, 1.0, -1.0, 2.0, 1.0, 1.0, -1.0, -1.0, -2.0, 1.0, -1.0, -1.0, -1.0, -1.0, -2.0, -2.0, 1.0, 1.0, 1.0, 1.0, 1.0, 1.0, -1.0, -1.0, -1.0, -1.0, -1.0, -1.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  static constexpr int T_CSR_SLOT[82][6] = {{0, 4, -1, 3, 5, -1}, {0, 5, -1, 2, 3, -1}, {0, -1, -1, 3, -1, -1}, {3, 6, -1, 0, 1, -1}, {3, 7, -1, 0, 6, -1}, {1, 3, -1, 4, 5, -1}, {4, -1, -1, 1, -1, -1}, {1, 3, -1, 6, -1, -1}, {3, 6, -1, 0, 1, -1}, {4, 6, -1, 1, 5, -1}, {5, 6, -1, 1, 2, -1}, {6, -1, -1, 1, 7, -1}, {6, -1, -1, 1, 7, -1}, {0, 5, -1, 2, 3, -1}, {2, 4, -1, 5, -1, -1}, {3, 5, -1, 2, -1, -1}, {5, 6, -1, 1, 2, -1}, {3, 7, -1, 2, 5, -1}, {5, 7, -1, 2, 6, -1}, {5, 7, -1, 2, 6, -1}, {3, 5, -1, -1, -1, -1}, {1, 3, -1, 4, 5, -1}, {0, 4, -1, 3, 5, -1}, {0, 5, -1, 2, 3, -1}, {0, -1, -1, 3, -1, -1}, {3, 4, -1, 5, -1, -1}, {3, 5, -1, 2, -1, -1}, {1, 3, -1, 6, -1, -1}, {3, 6, -1, 0, 1, -1}, {3, 6, -1, 5, -1, -1}, {3, 7, -1, 2, 5, -1}, {3, 7, -1, 0, 6, -1}, {3, 5, -1, -1, -1, -1}, {1, 3, -1, 4, 5, -1}, {0, 4, -1, 3, 5, -1}, {2, 4, -1, 5, -1, -1}, {4, -1, -1, 1, -1, -1}, {3, 4, -1, 5, -1, -1}, {4, 6, -1, 1, 5, -1}, {4, 7, -1, 5, 6, -1}, {1, 3, -1, 4, 5, -1}, {0, 4, -1, 3, 5, -1}, {0, 5, -1, 2, 3, -1}, {2, 4, -1, 5, -1, -1}, {3, 4, -1, 5, -1, -1}, {3, 5, -1, 2, -1, -1}, {3, 6, -1, 5, -1, -1}, {4, 6, -1, 1, 5, -1}, {5, 6, -1, 1, 2, -1}, {7, -1, -1, 5, -1, -1}, {3, 7, -1, 2, 5, -1}, {4, 7, -1, 5, 6, -1}, {5, 7, -1, 2, 6, -1}, {5, 7, -1, 2, 6, -1}, {3, 5, -1, -1, -1, -1}, {1, 3, -1, 6, -1, -1}, {3, 6, -1, 0, 1, -1}, {3, 6, -1, 5, -1, -1}, {4, 6, -1, 1, 5, -1}, {5, 6, -1, 1, 2, -1}, {6, -1, -1, 1, 7, -1}, {6, -1, -1, 1, 7, -1}, {3, 7, -1, 0, 6, -1}, {4, 7, -1, 5, 6, -1}, {5, 7, -1, 2, 6, -1}, {5, 7, -1, 2, 6, -1}, {6, -1, -1, 1, 7, -1}, {6, -1, -1, 1, 7, -1}, {7, -1, -1, 5, -1, -1}, {3, 7, -1, 2, 5, -1}, {3, 7, -1, 0, 6, -1}, {4, 7, -1, 5, 6, -1}, {5, 7, -1, 2, 6, -1}, {5, 7, -1, 2, 6, -1}, {-1, -1, -1, -1, -1, -1}, {-1, -1, -1, -1, -1, -1}, {-1, -1, -1, -1, -1, -1}, {-1, -1, -1, -1, -1, -1}, {-1, -1, -1, -1, -1, -1}, {-1, -1, -1, -1, -1, -1}, {-1, -1, -1, -1, -1, -1}, {-1, -1, -1, -1, -1, -1}};
  static constexpr int T_CSR_EFF[82] = {-1, -1, 0, -1, -1, -1, 0, 1, -1, -1, -1, -1, -1, -1, -1, 0, -1, -1, -1, -1, -1, -1, -1, -1, 0, 0, 0, 1, -1, -1, -1, -1, -1, -1, -1, -1, 0, 0, -1, -1, -1, -1, -1, -1, 0, 0, -1, -1, -1, 0, -1, -1, -1, -1, -1, 1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, 0, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1};
  // no lane-group tables: 2 H + 2 OH => 2 H2O: order above 3
  static constexpr bool G_OK = false;
};
}  // namespace mech
}  // namespace pelec
