/* Generated by geos-chem_amd/mechgen/emit_tables.py from mech/Hg.json -- do not edit. */
#pragma once

namespace unroll_Hg {
constexpr int LDS_FIELDS = 160, NLU_LDS = 129, NRATE_LDS = 20;
template <class R, class F>
__device__ __forceinline__ void fun(const double (&y)[32], R rate, F fix, double (&v)[32]) {
  v[0] = 0.0;
  v[1] = 0.0;
  v[2] = 0.0;
  v[3] = 0.0;
  v[4] = 0.0;
  v[5] = 0.0;
  v[6] = 0.0;
  v[7] = 0.0;
  v[8] = 0.0;
  v[9] = 0.0;
  v[10] = 0.0;
  v[11] = 0.0;
  v[12] = 0.0;
  v[13] = 0.0;
  v[14] = 0.0;
  v[15] = 0.0;
  v[16] = 0.0;
  v[17] = 0.0;
  v[18] = 0.0;
  v[19] = 0.0;
  v[20] = 0.0;
  v[21] = 0.0;
  v[22] = 0.0;
  v[23] = 0.0;
  v[24] = 0.0;
  v[25] = 0.0;
  v[26] = 0.0;
  v[27] = 0.0;
  v[28] = 0.0;
  v[29] = 0.0;
  v[30] = 0.0;
  v[31] = 0.0;
  const double k0 = rate(0);
  const double k1 = rate(1);
  const double k2 = rate(2);
  const double k3 = rate(3);
  const double k4 = rate(4);
  const double k5 = rate(5);
  const double k6 = rate(6);
  const double k7 = rate(7);
  const double k8 = rate(8);
  const double k9 = rate(9);
  const double k10 = rate(10);
  const double k11 = rate(11);
  __builtin_amdgcn_sched_barrier(0);
  const double k12 = rate(12);
  const double k13 = rate(13);
  const double k14 = rate(14);
  const double k15 = rate(15);
  const double k16 = rate(16);
  const double k17 = rate(17);
  const double k18 = rate(18);
  const double k19 = rate(19);
  const double k20 = rate(20);
  const double k21 = rate(21);
  const double k22 = rate(22);
  const double k23 = rate(23);
  __builtin_amdgcn_sched_barrier(0);
  { const double k = k0; double a = k; a *= y[29]; a *= fix(0);
    v[2] = fma(1.0, a, v[2]);
    v[4] = fma(1.0, a, v[4]);
    v[29] = fma(-1.0, a, v[29]);
    v[31] = fma(1.0, a, v[31]);
  }
  { const double k = k1; double a = k; a *= y[31];
    v[3] = fma(1.0, a, v[3]);
    v[29] = fma(1.0, a, v[29]);
    v[31] = fma(-1.0, a, v[31]);
  }
  { const double k = k2; double a = k; a *= y[31]; a *= fix(0);
    v[3] = fma(1.0, a, v[3]);
    v[29] = fma(1.0, a, v[29]);
    v[31] = fma(-1.0, a, v[31]);
  }
  { const double k = k3; double a = k; a *= y[31]; a *= fix(3);
    v[3] = fma(1.0, a, v[3]);
    v[29] = fma(1.0, a, v[29]);
    v[31] = fma(-1.0, a, v[31]);
  }
  { const double k = k4; double a = k; a *= y[31]; a *= fix(3);
    v[15] = fma(1.0, a, v[15]);
    v[31] = fma(-1.0, a, v[31]);
  }
  { const double k = k5; double a = k; a *= y[31]; a *= fix(6);
    v[22] = fma(1.0, a, v[22]);
    v[31] = fma(-1.0, a, v[31]);
  }
  { const double k = k6; double a = k; a *= y[31]; a *= fix(8);
    v[12] = fma(1.0, a, v[12]);
    v[31] = fma(-1.0, a, v[31]);
  }
  { const double k = k7; double a = k; a *= y[31]; a *= fix(7);
    v[13] = fma(1.0, a, v[13]);
    v[31] = fma(-1.0, a, v[31]);
  }
  { const double k = k8; double a = k; a *= y[31]; a *= fix(2);
    v[30] = fma(1.0, a, v[30]);
    v[31] = fma(-1.0, a, v[31]);
  }
  { const double k = k9; double a = k; a *= y[31]; a *= fix(0);
    v[17] = fma(1.0, a, v[17]);
    v[31] = fma(-1.0, a, v[31]);
  }
  { const double k = k10; double a = k; a *= y[21]; a *= fix(10);
    v[21] = fma(-1.0, a, v[21]);
    v[30] = fma(1.0, a, v[30]);
  }
  { const double k = k11; double a = k; a *= y[21]; a *= fix(9);
    v[21] = fma(-1.0, a, v[21]);
    v[31] = fma(1.0, a, v[31]);
  }
  const double k24 = rate(24);
  const double k25 = rate(25);
  const double k26 = rate(26);
  const double k27 = rate(27);
  const double k28 = rate(28);
  const double k29 = rate(29);
  const double k30 = rate(30);
  const double k31 = rate(31);
  const double k32 = rate(32);
  const double k33 = rate(33);
  const double k34 = rate(34);
  const double k35 = rate(35);
  __builtin_amdgcn_sched_barrier(0);
  { const double k = k12; double a = k; a *= y[31]; a *= fix(5);
    v[21] = fma(1.0, a, v[21]);
    v[31] = fma(-1.0, a, v[31]);
  }
  { const double k = k13; double a = k; a *= y[29]; a *= fix(1);
    v[2] = fma(1.0, a, v[2]);
    v[6] = fma(1.0, a, v[6]);
    v[26] = fma(1.0, a, v[26]);
    v[29] = fma(-1.0, a, v[29]);
  }
  { const double k = k14; double a = k; a *= y[26]; a *= fix(1);
    v[3] = fma(1.0, a, v[3]);
    v[26] = fma(-1.0, a, v[26]);
    v[29] = fma(1.0, a, v[29]);
  }
  { const double k = k15; double a = k; a *= y[26]; a *= fix(3);
    v[3] = fma(1.0, a, v[3]);
    v[26] = fma(-1.0, a, v[26]);
    v[29] = fma(1.0, a, v[29]);
  }
  { const double k = k16; double a = k; a *= y[26]; a *= fix(3);
    v[16] = fma(1.0, a, v[16]);
    v[26] = fma(-1.0, a, v[26]);
  }
  { const double k = k17; double a = k; a *= y[26]; a *= fix(6);
    v[24] = fma(1.0, a, v[24]);
    v[26] = fma(-1.0, a, v[26]);
  }
  { const double k = k18; double a = k; a *= y[26]; a *= fix(8);
    v[7] = fma(1.0, a, v[7]);
    v[26] = fma(-1.0, a, v[26]);
  }
  { const double k = k19; double a = k; a *= y[26]; a *= fix(7);
    v[8] = fma(1.0, a, v[8]);
    v[26] = fma(-1.0, a, v[26]);
  }
  { const double k = k20; double a = k; a *= y[26]; a *= fix(0);
    v[9] = fma(1.0, a, v[9]);
    v[26] = fma(-1.0, a, v[26]);
  }
  { const double k = k21; double a = k; a *= y[26]; a *= fix(2);
    v[25] = fma(1.0, a, v[25]);
    v[26] = fma(-1.0, a, v[26]);
  }
  { const double k = k22; double a = k; a *= y[26]; a *= fix(5);
    v[23] = fma(1.0, a, v[23]);
    v[26] = fma(-1.0, a, v[26]);
  }
  { const double k = k23; double a = k; a *= y[23]; a *= fix(10);
    v[23] = fma(-1.0, a, v[23]);
    v[25] = fma(1.0, a, v[25]);
  }
  const double k36 = rate(36);
  const double k37 = rate(37);
  const double k38 = rate(38);
  const double k39 = rate(39);
  const double k40 = rate(40);
  const double k41 = rate(41);
  const double k42 = rate(42);
  const double k43 = rate(43);
  const double k44 = rate(44);
  const double k45 = rate(45);
  const double k46 = rate(46);
  const double k47 = rate(47);
  __builtin_amdgcn_sched_barrier(0);
  { const double k = k24; double a = k; a *= y[23]; a *= fix(9);
    v[23] = fma(-1.0, a, v[23]);
    v[26] = fma(1.0, a, v[26]);
  }
  { const double k = k25; double a = k; a *= y[29]; a *= fix(2);
    v[2] = fma(1.0, a, v[2]);
    v[5] = fma(1.0, a, v[5]);
    v[28] = fma(1.0, a, v[28]);
    v[29] = fma(-1.0, a, v[29]);
  }
  { const double k = k26; double a = k; a *= y[28];
    v[3] = fma(1.0, a, v[3]);
    v[28] = fma(-1.0, a, v[28]);
    v[29] = fma(1.0, a, v[29]);
  }
  { const double k = k27; double a = k; a *= y[28]; a *= fix(3);
    v[14] = fma(1.0, a, v[14]);
    v[28] = fma(-1.0, a, v[28]);
  }
  { const double k = k28; double a = k; a *= y[28]; a *= fix(6);
    v[20] = fma(1.0, a, v[20]);
    v[28] = fma(-1.0, a, v[28]);
  }
  { const double k = k29; double a = k; a *= y[28]; a *= fix(8);
    v[10] = fma(1.0, a, v[10]);
    v[28] = fma(-1.0, a, v[28]);
  }
  { const double k = k30; double a = k; a *= y[28]; a *= fix(7);
    v[11] = fma(1.0, a, v[11]);
    v[28] = fma(-1.0, a, v[28]);
  }
  { const double k = k31; double a = k; a *= y[28]; a *= fix(0);
    v[4] = fma(1.0, a, v[4]);
    v[28] = fma(-1.0, a, v[28]);
    v[30] = fma(1.0, a, v[30]);
  }
  { const double k = k32; double a = k; a *= y[28]; a *= fix(2);
    v[19] = fma(1.0, a, v[19]);
    v[28] = fma(-1.0, a, v[28]);
  }
  { const double k = k33; double a = k; a *= y[28]; a *= fix(5);
    v[18] = fma(1.0, a, v[18]);
    v[28] = fma(-1.0, a, v[28]);
  }
  { const double k = k34; double a = k; a *= y[18]; a *= fix(10);
    v[18] = fma(-1.0, a, v[18]);
    v[19] = fma(1.0, a, v[19]);
  }
  { const double k = k35; double a = k; a *= y[18]; a *= fix(9);
    v[18] = fma(-1.0, a, v[18]);
    v[28] = fma(1.0, a, v[28]);
  }
  const double k48 = rate(48);
  const double k49 = rate(49);
  const double k50 = rate(50);
  const double k51 = rate(51);
  const double k52 = rate(52);
  const double k53 = rate(53);
  const double k54 = rate(54);
  const double k55 = rate(55);
  const double k56 = rate(56);
  const double k57 = rate(57);
  const double k58 = rate(58);
  const double k59 = rate(59);
  __builtin_amdgcn_sched_barrier(0);
  { const double k = k36; double a = k; a *= y[15];
    v[15] = fma(-1.0, a, v[15]);
    v[27] = fma(1.0, a, v[27]);
  }
  { const double k = k37; double a = k; a *= y[22];
    v[22] = fma(-1.0, a, v[22]);
    v[27] = fma(1.0, a, v[27]);
  }
  { const double k = k38; double a = k; a *= y[30];
    v[27] = fma(1.0, a, v[27]);
    v[30] = fma(-1.0, a, v[30]);
  }
  { const double k = k39; double a = k; a *= y[13];
    v[13] = fma(-1.0, a, v[13]);
    v[27] = fma(1.0, a, v[27]);
  }
  { const double k = k40; double a = k; a *= y[12];
    v[12] = fma(-1.0, a, v[12]);
    v[27] = fma(1.0, a, v[27]);
  }
  { const double k = k41; double a = k; a *= y[17];
    v[17] = fma(-1.0, a, v[17]);
    v[27] = fma(1.0, a, v[27]);
  }
  { const double k = k42; double a = k; a *= y[16];
    v[16] = fma(-1.0, a, v[16]);
    v[27] = fma(1.0, a, v[27]);
  }
  { const double k = k43; double a = k; a *= y[24];
    v[24] = fma(-1.0, a, v[24]);
    v[27] = fma(1.0, a, v[27]);
  }
  { const double k = k44; double a = k; a *= y[25];
    v[25] = fma(-1.0, a, v[25]);
    v[27] = fma(1.0, a, v[27]);
  }
  { const double k = k45; double a = k; a *= y[8];
    v[8] = fma(-1.0, a, v[8]);
    v[27] = fma(1.0, a, v[27]);
  }
  { const double k = k46; double a = k; a *= y[7];
    v[7] = fma(-1.0, a, v[7]);
    v[27] = fma(1.0, a, v[27]);
  }
  { const double k = k47; double a = k; a *= y[9];
    v[9] = fma(-1.0, a, v[9]);
    v[27] = fma(1.0, a, v[27]);
  }
  const double k60 = rate(60);
  const double k61 = rate(61);
  const double k62 = rate(62);
  const double k63 = rate(63);
  const double k64 = rate(64);
  const double k65 = rate(65);
  const double k66 = rate(66);
  const double k67 = rate(67);
  const double k68 = rate(68);
  const double k69 = rate(69);
  const double k70 = rate(70);
  const double k71 = rate(71);
  __builtin_amdgcn_sched_barrier(0);
  { const double k = k48; double a = k; a *= y[0];
    v[0] = fma(-1.0, a, v[0]);
    v[27] = fma(1.0, a, v[27]);
  }
  { const double k = k49; double a = k; a *= y[14];
    v[14] = fma(-1.0, a, v[14]);
    v[27] = fma(1.0, a, v[27]);
  }
  { const double k = k50; double a = k; a *= y[20];
    v[20] = fma(-1.0, a, v[20]);
    v[27] = fma(1.0, a, v[27]);
  }
  { const double k = k51; double a = k; a *= y[19];
    v[19] = fma(-1.0, a, v[19]);
    v[27] = fma(1.0, a, v[27]);
  }
  { const double k = k52; double a = k; a *= y[11];
    v[11] = fma(-1.0, a, v[11]);
    v[27] = fma(1.0, a, v[27]);
  }
  { const double k = k53; double a = k; a *= y[10];
    v[10] = fma(-1.0, a, v[10]);
    v[27] = fma(1.0, a, v[27]);
  }
  { const double k = k54; double a = k; a *= y[15];
    v[1] = fma(1.0, a, v[1]);
    v[15] = fma(-1.0, a, v[15]);
  }
  { const double k = k55; double a = k; a *= y[22];
    v[1] = fma(1.0, a, v[1]);
    v[22] = fma(-1.0, a, v[22]);
  }
  { const double k = k56; double a = k; a *= y[30];
    v[1] = fma(1.0, a, v[1]);
    v[30] = fma(-1.0, a, v[30]);
  }
  { const double k = k57; double a = k; a *= y[13];
    v[1] = fma(1.0, a, v[1]);
    v[13] = fma(-1.0, a, v[13]);
  }
  { const double k = k58; double a = k; a *= y[12];
    v[1] = fma(1.0, a, v[1]);
    v[12] = fma(-1.0, a, v[12]);
  }
  { const double k = k59; double a = k; a *= y[17];
    v[1] = fma(1.0, a, v[1]);
    v[17] = fma(-1.0, a, v[17]);
  }
  const double k72 = rate(72);
  const double k73 = rate(73);
  const double k74 = rate(74);
  const double k75 = rate(75);
  const double k76 = rate(76);
  const double k77 = rate(77);
  const double k78 = rate(78);
  const double k79 = rate(79);
  const double k80 = rate(80);
  const double k81 = rate(81);
  const double k82 = rate(82);
  const double k83 = rate(83);
  __builtin_amdgcn_sched_barrier(0);
  { const double k = k60; double a = k; a *= y[16];
    v[1] = fma(1.0, a, v[1]);
    v[16] = fma(-1.0, a, v[16]);
  }
  { const double k = k61; double a = k; a *= y[24];
    v[1] = fma(1.0, a, v[1]);
    v[24] = fma(-1.0, a, v[24]);
  }
  { const double k = k62; double a = k; a *= y[25];
    v[1] = fma(1.0, a, v[1]);
    v[25] = fma(-1.0, a, v[25]);
  }
  { const double k = k63; double a = k; a *= y[8];
    v[1] = fma(1.0, a, v[1]);
    v[8] = fma(-1.0, a, v[8]);
  }
  { const double k = k64; double a = k; a *= y[7];
    v[1] = fma(1.0, a, v[1]);
    v[7] = fma(-1.0, a, v[7]);
  }
  { const double k = k65; double a = k; a *= y[9];
    v[1] = fma(1.0, a, v[1]);
    v[9] = fma(-1.0, a, v[9]);
  }
  { const double k = k66; double a = k; a *= y[14];
    v[1] = fma(1.0, a, v[1]);
    v[14] = fma(-1.0, a, v[14]);
  }
  { const double k = k67; double a = k; a *= y[20];
    v[1] = fma(1.0, a, v[1]);
    v[20] = fma(-1.0, a, v[20]);
  }
  { const double k = k68; double a = k; a *= y[19];
    v[1] = fma(1.0, a, v[1]);
    v[19] = fma(-1.0, a, v[19]);
  }
  { const double k = k69; double a = k; a *= y[11];
    v[1] = fma(1.0, a, v[1]);
    v[11] = fma(-1.0, a, v[11]);
  }
  { const double k = k70; double a = k; a *= y[10];
    v[1] = fma(1.0, a, v[1]);
    v[10] = fma(-1.0, a, v[10]);
  }
  { const double k = k71; double a = k; 
  }
  const double k84 = rate(84);
  const double k85 = rate(85);
  const double k86 = rate(86);
  const double k87 = rate(87);
  const double k88 = rate(88);
  const double k89 = rate(89);
  const double k90 = rate(90);
  const double k91 = rate(91);
  const double k92 = rate(92);
  const double k93 = rate(93);
  __builtin_amdgcn_sched_barrier(0);
  { const double k = k72; double a = k; 
  }
  { const double k = k73; double a = k; 
  }
  { const double k = k74; double a = k; a *= y[31];
    v[3] = fma(1.0, a, v[3]);
    v[29] = fma(1.0, a, v[29]);
    v[31] = fma(-1.0, a, v[31]);
  }
  { const double k = k75; double a = k; a *= y[15];
    v[15] = fma(-1.0, a, v[15]);
    v[21] = fma(0.9, a, v[21]);
    v[31] = fma(0.1, a, v[31]);
  }
  { const double k = k76; double a = k; a *= y[22];
    v[3] = fma(0.67, a, v[3]);
    v[21] = fma(0.25, a, v[21]);
    v[22] = fma(-1.0, a, v[22]);
    v[29] = fma(0.67, a, v[29]);
    v[30] = fma(0.01, a, v[30]);
    v[31] = fma(0.07, a, v[31]);
  }
  { const double k = k77; double a = k; a *= y[30];
    v[3] = fma(0.49, a, v[3]);
    v[5] = fma(0.35, a, v[5]);
    v[28] = fma(0.35, a, v[28]);
    v[29] = fma(0.49, a, v[29]);
    v[30] = fma(-0.99, a, v[30]);
    v[31] = fma(0.15, a, v[31]);
  }
  { const double k = k78; double a = k; a *= y[17];
    v[3] = fma(0.4, a, v[3]);
    v[17] = fma(-1.0, a, v[17]);
    v[29] = fma(0.4, a, v[29]);
    v[31] = fma(0.6, a, v[31]);
  }
  { const double k = k79; double a = k; a *= y[13];
    v[3] = fma(1.0, a, v[3]);
    v[13] = fma(-1.0, a, v[13]);
    v[29] = fma(1.0, a, v[29]);
  }
  { const double k = k80; double a = k; a *= y[12];
    v[3] = fma(1.0, a, v[3]);
    v[12] = fma(-1.0, a, v[12]);
    v[29] = fma(1.0, a, v[29]);
  }
  { const double k = k81; double a = k; a *= y[16];
    v[16] = fma(-1.0, a, v[16]);
    v[23] = fma(0.9, a, v[23]);
    v[26] = fma(0.1, a, v[26]);
  }
  { const double k = k82; double a = k; a *= y[24];
    v[3] = fma(0.67, a, v[3]);
    v[23] = fma(0.25, a, v[23]);
    v[24] = fma(-1.0, a, v[24]);
    v[25] = fma(0.01, a, v[25]);
    v[26] = fma(0.07, a, v[26]);
    v[29] = fma(0.67, a, v[29]);
  }
  { const double k = k83; double a = k; a *= y[25];
    v[3] = fma(0.49, a, v[3]);
    v[5] = fma(0.35, a, v[5]);
    v[25] = fma(-0.99, a, v[25]);
    v[26] = fma(0.15, a, v[26]);
    v[28] = fma(0.35, a, v[28]);
    v[29] = fma(0.49, a, v[29]);
  }
  { const double k = k84; double a = k; a *= y[9];
    v[9] = fma(-1.0, a, v[9]);
    v[26] = fma(1.0, a, v[26]);
  }
  { const double k = k85; double a = k; a *= y[8];
    v[8] = fma(-1.0, a, v[8]);
    v[26] = fma(1.0, a, v[26]);
  }
  { const double k = k86; double a = k; a *= y[7];
    v[7] = fma(-1.0, a, v[7]);
    v[26] = fma(1.0, a, v[26]);
  }
  { const double k = k87; double a = k; a *= y[28];
    v[3] = fma(1.0, a, v[3]);
    v[28] = fma(-1.0, a, v[28]);
    v[29] = fma(1.0, a, v[29]);
  }
  { const double k = k88; double a = k; a *= y[14];
    v[14] = fma(-1.0, a, v[14]);
    v[18] = fma(0.9, a, v[18]);
    v[28] = fma(0.1, a, v[28]);
  }
  { const double k = k89; double a = k; a *= y[20];
    v[3] = fma(0.67, a, v[3]);
    v[18] = fma(0.25, a, v[18]);
    v[19] = fma(0.01, a, v[19]);
    v[20] = fma(-1.0, a, v[20]);
    v[28] = fma(0.07, a, v[28]);
    v[29] = fma(0.67, a, v[29]);
  }
  { const double k = k90; double a = k; a *= y[19];
    v[3] = fma(1.0, a, v[3]);
    v[19] = fma(-1.0, a, v[19]);
    v[29] = fma(1.0, a, v[29]);
  }
  { const double k = k91; double a = k; a *= y[11];
    v[11] = fma(-1.0, a, v[11]);
    v[28] = fma(1.0, a, v[28]);
  }
  { const double k = k92; double a = k; a *= y[10];
    v[10] = fma(-1.0, a, v[10]);
    v[28] = fma(1.0, a, v[28]);
  }
  { const double k = k93; double a = k; a *= y[27];
    v[3] = fma(1.0, a, v[3]);
    v[27] = fma(-1.0, a, v[27]);
    v[29] = fma(1.0, a, v[29]);
  }
}
template <class R, class F>
__device__ __forceinline__ void fun_partials(const double (&y)[32], R rate, F fix, double (&v)[32], double (&b)[91]) {
  v[0] = 0.0;
  v[1] = 0.0;
  v[2] = 0.0;
  v[3] = 0.0;
  v[4] = 0.0;
  v[5] = 0.0;
  v[6] = 0.0;
  v[7] = 0.0;
  v[8] = 0.0;
  v[9] = 0.0;
  v[10] = 0.0;
  v[11] = 0.0;
  v[12] = 0.0;
  v[13] = 0.0;
  v[14] = 0.0;
  v[15] = 0.0;
  v[16] = 0.0;
  v[17] = 0.0;
  v[18] = 0.0;
  v[19] = 0.0;
  v[20] = 0.0;
  v[21] = 0.0;
  v[22] = 0.0;
  v[23] = 0.0;
  v[24] = 0.0;
  v[25] = 0.0;
  v[26] = 0.0;
  v[27] = 0.0;
  v[28] = 0.0;
  v[29] = 0.0;
  v[30] = 0.0;
  v[31] = 0.0;
  const double k0 = rate(0);
  const double k1 = rate(1);
  const double k2 = rate(2);
  const double k3 = rate(3);
  const double k4 = rate(4);
  const double k5 = rate(5);
  const double k6 = rate(6);
  const double k7 = rate(7);
  const double k8 = rate(8);
  const double k9 = rate(9);
  const double k10 = rate(10);
  const double k11 = rate(11);
  __builtin_amdgcn_sched_barrier(0);
  const double k12 = rate(12);
  const double k13 = rate(13);
  const double k14 = rate(14);
  const double k15 = rate(15);
  const double k16 = rate(16);
  const double k17 = rate(17);
  const double k18 = rate(18);
  const double k19 = rate(19);
  const double k20 = rate(20);
  const double k21 = rate(21);
  const double k22 = rate(22);
  const double k23 = rate(23);
  __builtin_amdgcn_sched_barrier(0);
  { const double k = k0; double a = k; a *= y[29]; a *= fix(0);
    v[2] = fma(1.0, a, v[2]);
    v[4] = fma(1.0, a, v[4]);
    v[29] = fma(-1.0, a, v[29]);
    v[31] = fma(1.0, a, v[31]);
    b[0] = k; b[0] *= fix(0);
  }
  { const double k = k1; double a = k; a *= y[31];
    v[3] = fma(1.0, a, v[3]);
    v[29] = fma(1.0, a, v[29]);
    v[31] = fma(-1.0, a, v[31]);
    b[1] = k; 
  }
  { const double k = k2; double a = k; a *= y[31]; a *= fix(0);
    v[3] = fma(1.0, a, v[3]);
    v[29] = fma(1.0, a, v[29]);
    v[31] = fma(-1.0, a, v[31]);
    b[2] = k; b[2] *= fix(0);
  }
  { const double k = k3; double a = k; a *= y[31]; a *= fix(3);
    v[3] = fma(1.0, a, v[3]);
    v[29] = fma(1.0, a, v[29]);
    v[31] = fma(-1.0, a, v[31]);
    b[3] = k; b[3] *= fix(3);
  }
  { const double k = k4; double a = k; a *= y[31]; a *= fix(3);
    v[15] = fma(1.0, a, v[15]);
    v[31] = fma(-1.0, a, v[31]);
    b[4] = k; b[4] *= fix(3);
  }
  { const double k = k5; double a = k; a *= y[31]; a *= fix(6);
    v[22] = fma(1.0, a, v[22]);
    v[31] = fma(-1.0, a, v[31]);
    b[5] = k; b[5] *= fix(6);
  }
  { const double k = k6; double a = k; a *= y[31]; a *= fix(8);
    v[12] = fma(1.0, a, v[12]);
    v[31] = fma(-1.0, a, v[31]);
    b[6] = k; b[6] *= fix(8);
  }
  { const double k = k7; double a = k; a *= y[31]; a *= fix(7);
    v[13] = fma(1.0, a, v[13]);
    v[31] = fma(-1.0, a, v[31]);
    b[7] = k; b[7] *= fix(7);
  }
  { const double k = k8; double a = k; a *= y[31]; a *= fix(2);
    v[30] = fma(1.0, a, v[30]);
    v[31] = fma(-1.0, a, v[31]);
    b[8] = k; b[8] *= fix(2);
  }
  { const double k = k9; double a = k; a *= y[31]; a *= fix(0);
    v[17] = fma(1.0, a, v[17]);
    v[31] = fma(-1.0, a, v[31]);
    b[9] = k; b[9] *= fix(0);
  }
  { const double k = k10; double a = k; a *= y[21]; a *= fix(10);
    v[21] = fma(-1.0, a, v[21]);
    v[30] = fma(1.0, a, v[30]);
    b[10] = k; b[10] *= fix(10);
  }
  { const double k = k11; double a = k; a *= y[21]; a *= fix(9);
    v[21] = fma(-1.0, a, v[21]);
    v[31] = fma(1.0, a, v[31]);
    b[11] = k; b[11] *= fix(9);
  }
  const double k24 = rate(24);
  const double k25 = rate(25);
  const double k26 = rate(26);
  const double k27 = rate(27);
  const double k28 = rate(28);
  const double k29 = rate(29);
  const double k30 = rate(30);
  const double k31 = rate(31);
  const double k32 = rate(32);
  const double k33 = rate(33);
  const double k34 = rate(34);
  const double k35 = rate(35);
  __builtin_amdgcn_sched_barrier(0);
  { const double k = k12; double a = k; a *= y[31]; a *= fix(5);
    v[21] = fma(1.0, a, v[21]);
    v[31] = fma(-1.0, a, v[31]);
    b[12] = k; b[12] *= fix(5);
  }
  { const double k = k13; double a = k; a *= y[29]; a *= fix(1);
    v[2] = fma(1.0, a, v[2]);
    v[6] = fma(1.0, a, v[6]);
    v[26] = fma(1.0, a, v[26]);
    v[29] = fma(-1.0, a, v[29]);
    b[13] = k; b[13] *= fix(1);
  }
  { const double k = k14; double a = k; a *= y[26]; a *= fix(1);
    v[3] = fma(1.0, a, v[3]);
    v[26] = fma(-1.0, a, v[26]);
    v[29] = fma(1.0, a, v[29]);
    b[14] = k; b[14] *= fix(1);
  }
  { const double k = k15; double a = k; a *= y[26]; a *= fix(3);
    v[3] = fma(1.0, a, v[3]);
    v[26] = fma(-1.0, a, v[26]);
    v[29] = fma(1.0, a, v[29]);
    b[15] = k; b[15] *= fix(3);
  }
  { const double k = k16; double a = k; a *= y[26]; a *= fix(3);
    v[16] = fma(1.0, a, v[16]);
    v[26] = fma(-1.0, a, v[26]);
    b[16] = k; b[16] *= fix(3);
  }
  { const double k = k17; double a = k; a *= y[26]; a *= fix(6);
    v[24] = fma(1.0, a, v[24]);
    v[26] = fma(-1.0, a, v[26]);
    b[17] = k; b[17] *= fix(6);
  }
  { const double k = k18; double a = k; a *= y[26]; a *= fix(8);
    v[7] = fma(1.0, a, v[7]);
    v[26] = fma(-1.0, a, v[26]);
    b[18] = k; b[18] *= fix(8);
  }
  { const double k = k19; double a = k; a *= y[26]; a *= fix(7);
    v[8] = fma(1.0, a, v[8]);
    v[26] = fma(-1.0, a, v[26]);
    b[19] = k; b[19] *= fix(7);
  }
  { const double k = k20; double a = k; a *= y[26]; a *= fix(0);
    v[9] = fma(1.0, a, v[9]);
    v[26] = fma(-1.0, a, v[26]);
    b[20] = k; b[20] *= fix(0);
  }
  { const double k = k21; double a = k; a *= y[26]; a *= fix(2);
    v[25] = fma(1.0, a, v[25]);
    v[26] = fma(-1.0, a, v[26]);
    b[21] = k; b[21] *= fix(2);
  }
  { const double k = k22; double a = k; a *= y[26]; a *= fix(5);
    v[23] = fma(1.0, a, v[23]);
    v[26] = fma(-1.0, a, v[26]);
    b[22] = k; b[22] *= fix(5);
  }
  { const double k = k23; double a = k; a *= y[23]; a *= fix(10);
    v[23] = fma(-1.0, a, v[23]);
    v[25] = fma(1.0, a, v[25]);
    b[23] = k; b[23] *= fix(10);
  }
  const double k36 = rate(36);
  const double k37 = rate(37);
  const double k38 = rate(38);
  const double k39 = rate(39);
  const double k40 = rate(40);
  const double k41 = rate(41);
  const double k42 = rate(42);
  const double k43 = rate(43);
  const double k44 = rate(44);
  const double k45 = rate(45);
  const double k46 = rate(46);
  const double k47 = rate(47);
  __builtin_amdgcn_sched_barrier(0);
  { const double k = k24; double a = k; a *= y[23]; a *= fix(9);
    v[23] = fma(-1.0, a, v[23]);
    v[26] = fma(1.0, a, v[26]);
    b[24] = k; b[24] *= fix(9);
  }
  { const double k = k25; double a = k; a *= y[29]; a *= fix(2);
    v[2] = fma(1.0, a, v[2]);
    v[5] = fma(1.0, a, v[5]);
    v[28] = fma(1.0, a, v[28]);
    v[29] = fma(-1.0, a, v[29]);
    b[25] = k; b[25] *= fix(2);
  }
  { const double k = k26; double a = k; a *= y[28];
    v[3] = fma(1.0, a, v[3]);
    v[28] = fma(-1.0, a, v[28]);
    v[29] = fma(1.0, a, v[29]);
    b[26] = k; 
  }
  { const double k = k27; double a = k; a *= y[28]; a *= fix(3);
    v[14] = fma(1.0, a, v[14]);
    v[28] = fma(-1.0, a, v[28]);
    b[27] = k; b[27] *= fix(3);
  }
  { const double k = k28; double a = k; a *= y[28]; a *= fix(6);
    v[20] = fma(1.0, a, v[20]);
    v[28] = fma(-1.0, a, v[28]);
    b[28] = k; b[28] *= fix(6);
  }
  { const double k = k29; double a = k; a *= y[28]; a *= fix(8);
    v[10] = fma(1.0, a, v[10]);
    v[28] = fma(-1.0, a, v[28]);
    b[29] = k; b[29] *= fix(8);
  }
  { const double k = k30; double a = k; a *= y[28]; a *= fix(7);
    v[11] = fma(1.0, a, v[11]);
    v[28] = fma(-1.0, a, v[28]);
    b[30] = k; b[30] *= fix(7);
  }
  { const double k = k31; double a = k; a *= y[28]; a *= fix(0);
    v[4] = fma(1.0, a, v[4]);
    v[28] = fma(-1.0, a, v[28]);
    v[30] = fma(1.0, a, v[30]);
    b[31] = k; b[31] *= fix(0);
  }
  { const double k = k32; double a = k; a *= y[28]; a *= fix(2);
    v[19] = fma(1.0, a, v[19]);
    v[28] = fma(-1.0, a, v[28]);
    b[32] = k; b[32] *= fix(2);
  }
  { const double k = k33; double a = k; a *= y[28]; a *= fix(5);
    v[18] = fma(1.0, a, v[18]);
    v[28] = fma(-1.0, a, v[28]);
    b[33] = k; b[33] *= fix(5);
  }
  { const double k = k34; double a = k; a *= y[18]; a *= fix(10);
    v[18] = fma(-1.0, a, v[18]);
    v[19] = fma(1.0, a, v[19]);
    b[34] = k; b[34] *= fix(10);
  }
  { const double k = k35; double a = k; a *= y[18]; a *= fix(9);
    v[18] = fma(-1.0, a, v[18]);
    v[28] = fma(1.0, a, v[28]);
    b[35] = k; b[35] *= fix(9);
  }
  const double k48 = rate(48);
  const double k49 = rate(49);
  const double k50 = rate(50);
  const double k51 = rate(51);
  const double k52 = rate(52);
  const double k53 = rate(53);
  const double k54 = rate(54);
  const double k55 = rate(55);
  const double k56 = rate(56);
  const double k57 = rate(57);
  const double k58 = rate(58);
  const double k59 = rate(59);
  __builtin_amdgcn_sched_barrier(0);
  { const double k = k36; double a = k; a *= y[15];
    v[15] = fma(-1.0, a, v[15]);
    v[27] = fma(1.0, a, v[27]);
    b[36] = k; 
  }
  { const double k = k37; double a = k; a *= y[22];
    v[22] = fma(-1.0, a, v[22]);
    v[27] = fma(1.0, a, v[27]);
    b[37] = k; 
  }
  { const double k = k38; double a = k; a *= y[30];
    v[27] = fma(1.0, a, v[27]);
    v[30] = fma(-1.0, a, v[30]);
    b[38] = k; 
  }
  { const double k = k39; double a = k; a *= y[13];
    v[13] = fma(-1.0, a, v[13]);
    v[27] = fma(1.0, a, v[27]);
    b[39] = k; 
  }
  { const double k = k40; double a = k; a *= y[12];
    v[12] = fma(-1.0, a, v[12]);
    v[27] = fma(1.0, a, v[27]);
    b[40] = k; 
  }
  { const double k = k41; double a = k; a *= y[17];
    v[17] = fma(-1.0, a, v[17]);
    v[27] = fma(1.0, a, v[27]);
    b[41] = k; 
  }
  { const double k = k42; double a = k; a *= y[16];
    v[16] = fma(-1.0, a, v[16]);
    v[27] = fma(1.0, a, v[27]);
    b[42] = k; 
  }
  { const double k = k43; double a = k; a *= y[24];
    v[24] = fma(-1.0, a, v[24]);
    v[27] = fma(1.0, a, v[27]);
    b[43] = k; 
  }
  { const double k = k44; double a = k; a *= y[25];
    v[25] = fma(-1.0, a, v[25]);
    v[27] = fma(1.0, a, v[27]);
    b[44] = k; 
  }
  { const double k = k45; double a = k; a *= y[8];
    v[8] = fma(-1.0, a, v[8]);
    v[27] = fma(1.0, a, v[27]);
    b[45] = k; 
  }
  { const double k = k46; double a = k; a *= y[7];
    v[7] = fma(-1.0, a, v[7]);
    v[27] = fma(1.0, a, v[27]);
    b[46] = k; 
  }
  { const double k = k47; double a = k; a *= y[9];
    v[9] = fma(-1.0, a, v[9]);
    v[27] = fma(1.0, a, v[27]);
    b[47] = k; 
  }
  const double k60 = rate(60);
  const double k61 = rate(61);
  const double k62 = rate(62);
  const double k63 = rate(63);
  const double k64 = rate(64);
  const double k65 = rate(65);
  const double k66 = rate(66);
  const double k67 = rate(67);
  const double k68 = rate(68);
  const double k69 = rate(69);
  const double k70 = rate(70);
  const double k71 = rate(71);
  __builtin_amdgcn_sched_barrier(0);
  { const double k = k48; double a = k; a *= y[0];
    v[0] = fma(-1.0, a, v[0]);
    v[27] = fma(1.0, a, v[27]);
    b[48] = k; 
  }
  { const double k = k49; double a = k; a *= y[14];
    v[14] = fma(-1.0, a, v[14]);
    v[27] = fma(1.0, a, v[27]);
    b[49] = k; 
  }
  { const double k = k50; double a = k; a *= y[20];
    v[20] = fma(-1.0, a, v[20]);
    v[27] = fma(1.0, a, v[27]);
    b[50] = k; 
  }
  { const double k = k51; double a = k; a *= y[19];
    v[19] = fma(-1.0, a, v[19]);
    v[27] = fma(1.0, a, v[27]);
    b[51] = k; 
  }
  { const double k = k52; double a = k; a *= y[11];
    v[11] = fma(-1.0, a, v[11]);
    v[27] = fma(1.0, a, v[27]);
    b[52] = k; 
  }
  { const double k = k53; double a = k; a *= y[10];
    v[10] = fma(-1.0, a, v[10]);
    v[27] = fma(1.0, a, v[27]);
    b[53] = k; 
  }
  { const double k = k54; double a = k; a *= y[15];
    v[1] = fma(1.0, a, v[1]);
    v[15] = fma(-1.0, a, v[15]);
    b[54] = k; 
  }
  { const double k = k55; double a = k; a *= y[22];
    v[1] = fma(1.0, a, v[1]);
    v[22] = fma(-1.0, a, v[22]);
    b[55] = k; 
  }
  { const double k = k56; double a = k; a *= y[30];
    v[1] = fma(1.0, a, v[1]);
    v[30] = fma(-1.0, a, v[30]);
    b[56] = k; 
  }
  { const double k = k57; double a = k; a *= y[13];
    v[1] = fma(1.0, a, v[1]);
    v[13] = fma(-1.0, a, v[13]);
    b[57] = k; 
  }
  { const double k = k58; double a = k; a *= y[12];
    v[1] = fma(1.0, a, v[1]);
    v[12] = fma(-1.0, a, v[12]);
    b[58] = k; 
  }
  { const double k = k59; double a = k; a *= y[17];
    v[1] = fma(1.0, a, v[1]);
    v[17] = fma(-1.0, a, v[17]);
    b[59] = k; 
  }
  const double k72 = rate(72);
  const double k73 = rate(73);
  const double k74 = rate(74);
  const double k75 = rate(75);
  const double k76 = rate(76);
  const double k77 = rate(77);
  const double k78 = rate(78);
  const double k79 = rate(79);
  const double k80 = rate(80);
  const double k81 = rate(81);
  const double k82 = rate(82);
  const double k83 = rate(83);
  __builtin_amdgcn_sched_barrier(0);
  { const double k = k60; double a = k; a *= y[16];
    v[1] = fma(1.0, a, v[1]);
    v[16] = fma(-1.0, a, v[16]);
    b[60] = k; 
  }
  { const double k = k61; double a = k; a *= y[24];
    v[1] = fma(1.0, a, v[1]);
    v[24] = fma(-1.0, a, v[24]);
    b[61] = k; 
  }
  { const double k = k62; double a = k; a *= y[25];
    v[1] = fma(1.0, a, v[1]);
    v[25] = fma(-1.0, a, v[25]);
    b[62] = k; 
  }
  { const double k = k63; double a = k; a *= y[8];
    v[1] = fma(1.0, a, v[1]);
    v[8] = fma(-1.0, a, v[8]);
    b[63] = k; 
  }
  { const double k = k64; double a = k; a *= y[7];
    v[1] = fma(1.0, a, v[1]);
    v[7] = fma(-1.0, a, v[7]);
    b[64] = k; 
  }
  { const double k = k65; double a = k; a *= y[9];
    v[1] = fma(1.0, a, v[1]);
    v[9] = fma(-1.0, a, v[9]);
    b[65] = k; 
  }
  { const double k = k66; double a = k; a *= y[14];
    v[1] = fma(1.0, a, v[1]);
    v[14] = fma(-1.0, a, v[14]);
    b[66] = k; 
  }
  { const double k = k67; double a = k; a *= y[20];
    v[1] = fma(1.0, a, v[1]);
    v[20] = fma(-1.0, a, v[20]);
    b[67] = k; 
  }
  { const double k = k68; double a = k; a *= y[19];
    v[1] = fma(1.0, a, v[1]);
    v[19] = fma(-1.0, a, v[19]);
    b[68] = k; 
  }
  { const double k = k69; double a = k; a *= y[11];
    v[1] = fma(1.0, a, v[1]);
    v[11] = fma(-1.0, a, v[11]);
    b[69] = k; 
  }
  { const double k = k70; double a = k; a *= y[10];
    v[1] = fma(1.0, a, v[1]);
    v[10] = fma(-1.0, a, v[10]);
    b[70] = k; 
  }
  { const double k = k71; double a = k; 
  }
  const double k84 = rate(84);
  const double k85 = rate(85);
  const double k86 = rate(86);
  const double k87 = rate(87);
  const double k88 = rate(88);
  const double k89 = rate(89);
  const double k90 = rate(90);
  const double k91 = rate(91);
  const double k92 = rate(92);
  const double k93 = rate(93);
  __builtin_amdgcn_sched_barrier(0);
  { const double k = k72; double a = k; 
  }
  { const double k = k73; double a = k; 
  }
  { const double k = k74; double a = k; a *= y[31];
    v[3] = fma(1.0, a, v[3]);
    v[29] = fma(1.0, a, v[29]);
    v[31] = fma(-1.0, a, v[31]);
    b[71] = k; 
  }
  { const double k = k75; double a = k; a *= y[15];
    v[15] = fma(-1.0, a, v[15]);
    v[21] = fma(0.9, a, v[21]);
    v[31] = fma(0.1, a, v[31]);
    b[72] = k; 
  }
  { const double k = k76; double a = k; a *= y[22];
    v[3] = fma(0.67, a, v[3]);
    v[21] = fma(0.25, a, v[21]);
    v[22] = fma(-1.0, a, v[22]);
    v[29] = fma(0.67, a, v[29]);
    v[30] = fma(0.01, a, v[30]);
    v[31] = fma(0.07, a, v[31]);
    b[73] = k; 
  }
  { const double k = k77; double a = k; a *= y[30];
    v[3] = fma(0.49, a, v[3]);
    v[5] = fma(0.35, a, v[5]);
    v[28] = fma(0.35, a, v[28]);
    v[29] = fma(0.49, a, v[29]);
    v[30] = fma(-0.99, a, v[30]);
    v[31] = fma(0.15, a, v[31]);
    b[74] = k; 
  }
  { const double k = k78; double a = k; a *= y[17];
    v[3] = fma(0.4, a, v[3]);
    v[17] = fma(-1.0, a, v[17]);
    v[29] = fma(0.4, a, v[29]);
    v[31] = fma(0.6, a, v[31]);
    b[75] = k; 
  }
  { const double k = k79; double a = k; a *= y[13];
    v[3] = fma(1.0, a, v[3]);
    v[13] = fma(-1.0, a, v[13]);
    v[29] = fma(1.0, a, v[29]);
    b[76] = k; 
  }
  { const double k = k80; double a = k; a *= y[12];
    v[3] = fma(1.0, a, v[3]);
    v[12] = fma(-1.0, a, v[12]);
    v[29] = fma(1.0, a, v[29]);
    b[77] = k; 
  }
  { const double k = k81; double a = k; a *= y[16];
    v[16] = fma(-1.0, a, v[16]);
    v[23] = fma(0.9, a, v[23]);
    v[26] = fma(0.1, a, v[26]);
    b[78] = k; 
  }
  { const double k = k82; double a = k; a *= y[24];
    v[3] = fma(0.67, a, v[3]);
    v[23] = fma(0.25, a, v[23]);
    v[24] = fma(-1.0, a, v[24]);
    v[25] = fma(0.01, a, v[25]);
    v[26] = fma(0.07, a, v[26]);
    v[29] = fma(0.67, a, v[29]);
    b[79] = k; 
  }
  { const double k = k83; double a = k; a *= y[25];
    v[3] = fma(0.49, a, v[3]);
    v[5] = fma(0.35, a, v[5]);
    v[25] = fma(-0.99, a, v[25]);
    v[26] = fma(0.15, a, v[26]);
    v[28] = fma(0.35, a, v[28]);
    v[29] = fma(0.49, a, v[29]);
    b[80] = k; 
  }
  { const double k = k84; double a = k; a *= y[9];
    v[9] = fma(-1.0, a, v[9]);
    v[26] = fma(1.0, a, v[26]);
    b[81] = k; 
  }
  { const double k = k85; double a = k; a *= y[8];
    v[8] = fma(-1.0, a, v[8]);
    v[26] = fma(1.0, a, v[26]);
    b[82] = k; 
  }
  { const double k = k86; double a = k; a *= y[7];
    v[7] = fma(-1.0, a, v[7]);
    v[26] = fma(1.0, a, v[26]);
    b[83] = k; 
  }
  { const double k = k87; double a = k; a *= y[28];
    v[3] = fma(1.0, a, v[3]);
    v[28] = fma(-1.0, a, v[28]);
    v[29] = fma(1.0, a, v[29]);
    b[84] = k; 
  }
  { const double k = k88; double a = k; a *= y[14];
    v[14] = fma(-1.0, a, v[14]);
    v[18] = fma(0.9, a, v[18]);
    v[28] = fma(0.1, a, v[28]);
    b[85] = k; 
  }
  { const double k = k89; double a = k; a *= y[20];
    v[3] = fma(0.67, a, v[3]);
    v[18] = fma(0.25, a, v[18]);
    v[19] = fma(0.01, a, v[19]);
    v[20] = fma(-1.0, a, v[20]);
    v[28] = fma(0.07, a, v[28]);
    v[29] = fma(0.67, a, v[29]);
    b[86] = k; 
  }
  { const double k = k90; double a = k; a *= y[19];
    v[3] = fma(1.0, a, v[3]);
    v[19] = fma(-1.0, a, v[19]);
    v[29] = fma(1.0, a, v[29]);
    b[87] = k; 
  }
  { const double k = k91; double a = k; a *= y[11];
    v[11] = fma(-1.0, a, v[11]);
    v[28] = fma(1.0, a, v[28]);
    b[88] = k; 
  }
  { const double k = k92; double a = k; a *= y[10];
    v[10] = fma(-1.0, a, v[10]);
    v[28] = fma(1.0, a, v[28]);
    b[89] = k; 
  }
  { const double k = k93; double a = k; a *= y[27];
    v[3] = fma(1.0, a, v[3]);
    v[27] = fma(-1.0, a, v[27]);
    v[29] = fma(1.0, a, v[29]);
    b[90] = k; 
  }
}
template <class LG, class LP>
__device__ __forceinline__ bool lu(const double (&b)[91], double diag, double (&d)[32], LG lds, LP put_lds) {
  bool bad = false;
  { double g = 0.0;
    g = fma(1.0, b[48], g);
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[0] = g; }
  { double g = 0.0;
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[1] = g; }
  { double g = 0.0;
    g = fma(-1.0, b[64], g);
    put_lds(0, g); }
  { double g = 0.0;
    g = fma(-1.0, b[63], g);
    put_lds(1, g); }
  { double g = 0.0;
    g = fma(-1.0, b[65], g);
    put_lds(2, g); }
  { double g = 0.0;
    g = fma(-1.0, b[70], g);
    put_lds(3, g); }
  { double g = 0.0;
    g = fma(-1.0, b[69], g);
    put_lds(4, g); }
  { double g = 0.0;
    g = fma(-1.0, b[58], g);
    put_lds(5, g); }
  { double g = 0.0;
    g = fma(-1.0, b[57], g);
    put_lds(6, g); }
  { double g = 0.0;
    g = fma(-1.0, b[66], g);
    put_lds(7, g); }
  { double g = 0.0;
    g = fma(-1.0, b[54], g);
    put_lds(8, g); }
  { double g = 0.0;
    g = fma(-1.0, b[60], g);
    put_lds(9, g); }
  { double g = 0.0;
    g = fma(-1.0, b[59], g);
    put_lds(10, g); }
  { double g = 0.0;
    g = fma(-1.0, b[68], g);
    put_lds(11, g); }
  { double g = 0.0;
    g = fma(-1.0, b[67], g);
    put_lds(12, g); }
  { double g = 0.0;
    g = fma(-1.0, b[55], g);
    put_lds(13, g); }
  { double g = 0.0;
    g = fma(-1.0, b[61], g);
    put_lds(14, g); }
  { double g = 0.0;
    g = fma(-1.0, b[62], g);
    put_lds(15, g); }
  { double g = 0.0;
    g = fma(-1.0, b[56], g);
    put_lds(16, g); }
  { double g = 0.0;
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[2] = g; }
  { double g = 0.0;
    g = fma(-1.0, b[0], g);
    g = fma(-1.0, b[13], g);
    g = fma(-1.0, b[25], g);
    put_lds(17, g); }
  { double g = 0.0;
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[3] = g; }
  { double g = 0.0;
    g = fma(-1.0, b[77], g);
    put_lds(18, g); }
  { double g = 0.0;
    g = fma(-1.0, b[76], g);
    put_lds(19, g); }
  { double g = 0.0;
    g = fma(-0.4, b[75], g);
    put_lds(20, g); }
  { double g = 0.0;
    g = fma(-1.0, b[87], g);
    put_lds(21, g); }
  { double g = 0.0;
    g = fma(-0.67, b[86], g);
    put_lds(22, g); }
  { double g = 0.0;
    g = fma(-0.67, b[73], g);
    put_lds(23, g); }
  { double g = 0.0;
    g = fma(-0.67, b[79], g);
    put_lds(24, g); }
  { double g = 0.0;
    g = fma(-0.49, b[80], g);
    put_lds(25, g); }
  { double g = 0.0;
    g = fma(-1.0, b[14], g);
    g = fma(-1.0, b[15], g);
    put_lds(26, g); }
  { double g = 0.0;
    g = fma(-1.0, b[90], g);
    put_lds(27, g); }
  { double g = 0.0;
    g = fma(-1.0, b[26], g);
    g = fma(-1.0, b[84], g);
    put_lds(28, g); }
  { double g = 0.0;
    g = fma(-0.49, b[74], g);
    put_lds(29, g); }
  { double g = 0.0;
    g = fma(-1.0, b[1], g);
    g = fma(-1.0, b[2], g);
    g = fma(-1.0, b[3], g);
    g = fma(-1.0, b[71], g);
    put_lds(30, g); }
  { double g = 0.0;
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[4] = g; }
  { double g = 0.0;
    g = fma(-1.0, b[31], g);
    put_lds(31, g); }
  { double g = 0.0;
    g = fma(-1.0, b[0], g);
    put_lds(32, g); }
  { double g = 0.0;
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[5] = g; }
  { double g = 0.0;
    g = fma(-0.35, b[80], g);
    put_lds(33, g); }
  { double g = 0.0;
    g = fma(-1.0, b[25], g);
    put_lds(34, g); }
  { double g = 0.0;
    g = fma(-0.35, b[74], g);
    put_lds(35, g); }
  { double g = 0.0;
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[6] = g; }
  { double g = 0.0;
    g = fma(-1.0, b[13], g);
    put_lds(36, g); }
  { double g = 0.0;
    g = fma(1.0, b[46], g);
    g = fma(1.0, b[64], g);
    g = fma(1.0, b[83], g);
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[7] = g; }
  { double g = 0.0;
    g = fma(-1.0, b[18], g);
    put_lds(37, g); }
  { double g = 0.0;
    g = fma(1.0, b[45], g);
    g = fma(1.0, b[63], g);
    g = fma(1.0, b[82], g);
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[8] = g; }
  { double g = 0.0;
    g = fma(-1.0, b[19], g);
    put_lds(38, g); }
  { double g = 0.0;
    g = fma(1.0, b[47], g);
    g = fma(1.0, b[65], g);
    g = fma(1.0, b[81], g);
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[9] = g; }
  { double g = 0.0;
    g = fma(-1.0, b[20], g);
    put_lds(39, g); }
  { double g = 0.0;
    g = fma(1.0, b[53], g);
    g = fma(1.0, b[70], g);
    g = fma(1.0, b[89], g);
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[10] = g; }
  { double g = 0.0;
    g = fma(-1.0, b[29], g);
    put_lds(40, g); }
  { double g = 0.0;
    g = fma(1.0, b[52], g);
    g = fma(1.0, b[69], g);
    g = fma(1.0, b[88], g);
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[11] = g; }
  { double g = 0.0;
    g = fma(-1.0, b[30], g);
    put_lds(41, g); }
  { double g = 0.0;
    g = fma(1.0, b[40], g);
    g = fma(1.0, b[58], g);
    g = fma(1.0, b[77], g);
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[12] = g; }
  { double g = 0.0;
    g = fma(-1.0, b[6], g);
    put_lds(42, g); }
  { double g = 0.0;
    g = fma(1.0, b[39], g);
    g = fma(1.0, b[57], g);
    g = fma(1.0, b[76], g);
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[13] = g; }
  { double g = 0.0;
    g = fma(-1.0, b[7], g);
    put_lds(43, g); }
  { double g = 0.0;
    g = fma(1.0, b[49], g);
    g = fma(1.0, b[66], g);
    g = fma(1.0, b[85], g);
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[14] = g; }
  { double g = 0.0;
    g = fma(-1.0, b[27], g);
    put_lds(44, g); }
  { double g = 0.0;
    g = fma(1.0, b[36], g);
    g = fma(1.0, b[54], g);
    g = fma(1.0, b[72], g);
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[15] = g; }
  { double g = 0.0;
    g = fma(-1.0, b[4], g);
    put_lds(45, g); }
  { double g = 0.0;
    g = fma(1.0, b[42], g);
    g = fma(1.0, b[60], g);
    g = fma(1.0, b[78], g);
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[16] = g; }
  { double g = 0.0;
    g = fma(-1.0, b[16], g);
    put_lds(46, g); }
  { double g = 0.0;
    g = fma(1.0, b[41], g);
    g = fma(1.0, b[59], g);
    g = fma(1.0, b[75], g);
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[17] = g; }
  { double g = 0.0;
    g = fma(-1.0, b[9], g);
    put_lds(47, g); }
  { double g = 0.0;
    g = fma(-0.9, b[85], g);
    g = g / d[14];
    put_lds(48, g); }
  { double g = 0.0;
    g = fma(1.0, b[34], g);
    g = fma(1.0, b[35], g);
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[18] = g; }
  { double g = 0.0;
    g = fma(-0.25, b[86], g);
    put_lds(49, g); }
  { double g = 0.0;
    g = fma(-1.0, b[33], g);
    g = fma(-lds(48), lds(44), g);
    put_lds(50, g); }
  { double g = 0.0;
    g = fma(-1.0, b[34], g);
    g = g / d[18];
    put_lds(51, g); }
  { double g = 0.0;
    g = fma(1.0, b[51], g);
    g = fma(1.0, b[68], g);
    g = fma(1.0, b[87], g);
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[19] = g; }
  { double g = 0.0;
    g = fma(-0.01, b[86], g);
    g = fma(-lds(51), lds(49), g);
    put_lds(52, g); }
  { double g = 0.0;
    g = fma(-1.0, b[32], g);
    g = fma(-lds(51), lds(50), g);
    put_lds(53, g); }
  { double g = 0.0;
    g = fma(1.0, b[50], g);
    g = fma(1.0, b[67], g);
    g = fma(1.0, b[86], g);
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[20] = g; }
  { double g = 0.0;
    g = fma(-1.0, b[28], g);
    put_lds(54, g); }
  { double g = 0.0;
    g = fma(-0.9, b[72], g);
    g = g / d[15];
    put_lds(55, g); }
  { double g = 0.0;
    g = fma(1.0, b[10], g);
    g = fma(1.0, b[11], g);
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[21] = g; }
  { double g = 0.0;
    g = fma(-0.25, b[73], g);
    put_lds(56, g); }
  { double g = 0.0;
    g = fma(-1.0, b[12], g);
    g = fma(-lds(55), lds(45), g);
    put_lds(57, g); }
  { double g = 0.0;
    g = fma(1.0, b[37], g);
    g = fma(1.0, b[55], g);
    g = fma(1.0, b[73], g);
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[22] = g; }
  { double g = 0.0;
    g = fma(-1.0, b[5], g);
    put_lds(58, g); }
  { double g = 0.0;
    g = fma(-0.9, b[78], g);
    g = g / d[16];
    put_lds(59, g); }
  { double g = 0.0;
    g = fma(1.0, b[23], g);
    g = fma(1.0, b[24], g);
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[23] = g; }
  { double g = 0.0;
    g = fma(-0.25, b[79], g);
    put_lds(60, g); }
  { double g = 0.0;
    g = fma(-1.0, b[22], g);
    g = fma(-lds(59), lds(46), g);
    put_lds(61, g); }
  { double g = 0.0;
    g = fma(1.0, b[43], g);
    g = fma(1.0, b[61], g);
    g = fma(1.0, b[79], g);
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[24] = g; }
  { double g = 0.0;
    g = fma(-1.0, b[17], g);
    put_lds(62, g); }
  { double g = 0.0;
    g = fma(-1.0, b[23], g);
    g = g / d[23];
    put_lds(63, g); }
  { double g = 0.0;
    g = fma(-0.01, b[79], g);
    g = fma(-lds(63), lds(60), g);
    g = g / d[24];
    put_lds(64, g); }
  { double g = 0.0;
    g = fma(1.0, b[44], g);
    g = fma(1.0, b[62], g);
    g = fma(0.99, b[80], g);
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[25] = g; }
  { double g = 0.0;
    g = fma(-1.0, b[21], g);
    g = fma(-lds(63), lds(61), g);
    g = fma(-lds(64), lds(62), g);
    put_lds(65, g); }
  { double g = 0.0;
    g = fma(-1.0, b[83], g);
    g = g / d[7];
    put_lds(66, g); }
  { double g = 0.0;
    g = fma(-1.0, b[82], g);
    g = g / d[8];
    put_lds(67, g); }
  { double g = 0.0;
    g = fma(-1.0, b[81], g);
    g = g / d[9];
    put_lds(68, g); }
  { double g = 0.0;
    g = fma(-0.1, b[78], g);
    g = g / d[16];
    put_lds(69, g); }
  { double g = 0.0;
    g = fma(-1.0, b[24], g);
    g = g / d[23];
    put_lds(70, g); }
  { double g = 0.0;
    g = fma(-0.07, b[79], g);
    g = fma(-lds(70), lds(60), g);
    g = g / d[24];
    put_lds(71, g); }
  { double g = 0.0;
    g = fma(-0.15, b[80], g);
    g = g / d[25];
    put_lds(72, g); }
  { double g = 0.0;
    g = fma(1.0, b[14], g);
    g = fma(1.0, b[15], g);
    g = fma(1.0, b[16], g);
    g = fma(1.0, b[17], g);
    g = fma(1.0, b[18], g);
    g = fma(1.0, b[19], g);
    g = fma(1.0, b[20], g);
    g = fma(1.0, b[21], g);
    g = fma(1.0, b[22], g);
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    g = fma(-lds(66), lds(37), g);
    g = fma(-lds(67), lds(38), g);
    g = fma(-lds(68), lds(39), g);
    g = fma(-lds(69), lds(46), g);
    g = fma(-lds(70), lds(61), g);
    g = fma(-lds(71), lds(62), g);
    g = fma(-lds(72), lds(65), g);
    d[26] = g; }
  { double g = 0.0;
    g = fma(-1.0, b[13], g);
    put_lds(73, g); }
  { double g = 0.0;
    g = fma(-1.0, b[48], g);
    g = g / d[0];
    put_lds(74, g); }
  { double g = 0.0;
    g = fma(-1.0, b[46], g);
    g = g / d[7];
    put_lds(75, g); }
  { double g = 0.0;
    g = fma(-1.0, b[45], g);
    g = g / d[8];
    put_lds(76, g); }
  { double g = 0.0;
    g = fma(-1.0, b[47], g);
    g = g / d[9];
    put_lds(77, g); }
  { double g = 0.0;
    g = fma(-1.0, b[53], g);
    g = g / d[10];
    put_lds(78, g); }
  { double g = 0.0;
    g = fma(-1.0, b[52], g);
    g = g / d[11];
    put_lds(79, g); }
  { double g = 0.0;
    g = fma(-1.0, b[40], g);
    g = g / d[12];
    put_lds(80, g); }
  { double g = 0.0;
    g = fma(-1.0, b[39], g);
    g = g / d[13];
    put_lds(81, g); }
  { double g = 0.0;
    g = fma(-1.0, b[49], g);
    g = g / d[14];
    put_lds(82, g); }
  { double g = 0.0;
    g = fma(-1.0, b[36], g);
    g = g / d[15];
    put_lds(83, g); }
  { double g = 0.0;
    g = fma(-1.0, b[42], g);
    g = g / d[16];
    put_lds(84, g); }
  { double g = 0.0;
    g = fma(-1.0, b[41], g);
    g = g / d[17];
    put_lds(85, g); }
  { double g = 0.0;
    g = fma(-1.0, b[51], g);
    g = g / d[19];
    put_lds(86, g); }
  { double g = 0.0;
    g = fma(-1.0, b[50], g);
    g = fma(-lds(86), lds(52), g);
    g = g / d[20];
    put_lds(87, g); }
  { double g = 0.0;
    g = fma(-1.0, b[37], g);
    g = g / d[22];
    put_lds(88, g); }
  { double g = 0.0;
    g = fma(-1.0, b[43], g);
    g = g / d[24];
    put_lds(89, g); }
  { double g = 0.0;
    g = fma(-1.0, b[44], g);
    g = g / d[25];
    put_lds(90, g); }
  { double g = 0.0;
    g = fma(-lds(75), lds(37), g);
    g = fma(-lds(76), lds(38), g);
    g = fma(-lds(77), lds(39), g);
    g = fma(-lds(84), lds(46), g);
    g = fma(-lds(89), lds(62), g);
    g = fma(-lds(90), lds(65), g);
    g = g / d[26];
    put_lds(91, g); }
  { double g = 0.0;
    g = fma(1.0, b[90], g);
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    d[27] = g; }
  { double g = 0.0;
    g = fma(-lds(78), lds(40), g);
    g = fma(-lds(79), lds(41), g);
    g = fma(-lds(82), lds(44), g);
    g = fma(-lds(86), lds(53), g);
    g = fma(-lds(87), lds(54), g);
    put_lds(92, g); }
  { double g = 0.0;
    g = fma(-lds(91), lds(73), g);
    put_lds(93, g); }
  { double g = 0.0;
    g = fma(-1.0, b[38], g);
    put_lds(94, g); }
  { double g = 0.0;
    g = fma(-lds(80), lds(42), g);
    g = fma(-lds(81), lds(43), g);
    g = fma(-lds(83), lds(45), g);
    g = fma(-lds(85), lds(47), g);
    g = fma(-lds(88), lds(58), g);
    put_lds(95, g); }
  { double g = 0.0;
    g = fma(-1.0, b[89], g);
    g = g / d[10];
    put_lds(96, g); }
  { double g = 0.0;
    g = fma(-1.0, b[88], g);
    g = g / d[11];
    put_lds(97, g); }
  { double g = 0.0;
    g = fma(-0.1, b[85], g);
    g = g / d[14];
    put_lds(98, g); }
  { double g = 0.0;
    g = fma(-1.0, b[35], g);
    g = g / d[18];
    put_lds(99, g); }
  { double g = 0.0;
    g = fma(-0.07, b[86], g);
    g = fma(-lds(99), lds(49), g);
    g = g / d[20];
    put_lds(100, g); }
  { double g = 0.0;
    g = fma(-0.35, b[80], g);
    g = g / d[25];
    put_lds(101, g); }
  { double g = 0.0;
    g = fma(-lds(101), lds(65), g);
    g = g / d[26];
    put_lds(102, g); }
  { double g = 0.0;
    g = fma(1.0, b[26], g);
    g = fma(1.0, b[27], g);
    g = fma(1.0, b[28], g);
    g = fma(1.0, b[29], g);
    g = fma(1.0, b[30], g);
    g = fma(1.0, b[31], g);
    g = fma(1.0, b[32], g);
    g = fma(1.0, b[33], g);
    g = fma(1.0, b[84], g);
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    g = fma(-lds(96), lds(40), g);
    g = fma(-lds(97), lds(41), g);
    g = fma(-lds(98), lds(44), g);
    g = fma(-lds(99), lds(50), g);
    g = fma(-lds(100), lds(54), g);
    d[28] = g; }
  { double g = 0.0;
    g = fma(-1.0, b[25], g);
    g = fma(-lds(102), lds(73), g);
    put_lds(103, g); }
  { double g = 0.0;
    g = fma(-0.35, b[74], g);
    put_lds(104, g); }
  { double g = 0.0;
    g = fma(-1.0, b[77], g);
    g = g / d[12];
    put_lds(105, g); }
  { double g = 0.0;
    g = fma(-1.0, b[76], g);
    g = g / d[13];
    put_lds(106, g); }
  { double g = 0.0;
    g = fma(-0.4, b[75], g);
    g = g / d[17];
    put_lds(107, g); }
  { double g = 0.0;
    g = fma(-1.0, b[87], g);
    g = g / d[19];
    put_lds(108, g); }
  { double g = 0.0;
    g = fma(-0.67, b[86], g);
    g = fma(-lds(108), lds(52), g);
    g = g / d[20];
    put_lds(109, g); }
  { double g = 0.0;
    g = fma(-0.67, b[73], g);
    g = g / d[22];
    put_lds(110, g); }
  { double g = 0.0;
    g = fma(-0.67, b[79], g);
    g = g / d[24];
    put_lds(111, g); }
  { double g = 0.0;
    g = fma(-0.49, b[80], g);
    g = g / d[25];
    put_lds(112, g); }
  { double g = 0.0;
    g = fma(-1.0, b[14], g);
    g = fma(-1.0, b[15], g);
    g = fma(-lds(111), lds(62), g);
    g = fma(-lds(112), lds(65), g);
    g = g / d[26];
    put_lds(113, g); }
  { double g = 0.0;
    g = fma(-1.0, b[90], g);
    g = g / d[27];
    put_lds(114, g); }
  { double g = 0.0;
    g = fma(-1.0, b[26], g);
    g = fma(-1.0, b[84], g);
    g = fma(-lds(108), lds(53), g);
    g = fma(-lds(109), lds(54), g);
    g = fma(-lds(114), lds(92), g);
    g = g / d[28];
    put_lds(115, g); }
  { double g = 0.0;
    g = fma(1.0, b[0], g);
    g = fma(1.0, b[13], g);
    g = fma(1.0, b[25], g);
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    g = fma(-lds(113), lds(73), g);
    g = fma(-lds(114), lds(93), g);
    g = fma(-lds(115), lds(103), g);
    d[29] = g; }
  { double g = 0.0;
    g = fma(-0.49, b[74], g);
    g = fma(-lds(114), lds(94), g);
    g = fma(-lds(115), lds(104), g);
    put_lds(116, g); }
  { double g = 0.0;
    g = fma(-1.0, b[1], g);
    g = fma(-1.0, b[2], g);
    g = fma(-1.0, b[3], g);
    g = fma(-1.0, b[71], g);
    g = fma(-lds(105), lds(42), g);
    g = fma(-lds(106), lds(43), g);
    g = fma(-lds(107), lds(47), g);
    g = fma(-lds(110), lds(58), g);
    g = fma(-lds(114), lds(95), g);
    put_lds(117, g); }
  { double g = 0.0;
    g = fma(-1.0, b[10], g);
    g = g / d[21];
    put_lds(118, g); }
  { double g = 0.0;
    g = fma(-0.01, b[73], g);
    g = fma(-lds(118), lds(56), g);
    g = g / d[22];
    put_lds(119, g); }
  { double g = 0.0;
    g = fma(-1.0, b[31], g);
    g = g / d[28];
    put_lds(120, g); }
  { double g = 0.0;
    g = fma(-lds(120), lds(103), g);
    g = g / d[29];
    put_lds(121, g); }
  { double g = 0.0;
    g = fma(1.0, b[38], g);
    g = fma(1.0, b[56], g);
    g = fma(0.99, b[74], g);
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    g = fma(-lds(120), lds(104), g);
    g = fma(-lds(121), lds(116), g);
    d[30] = g; }
  { double g = 0.0;
    g = fma(-1.0, b[8], g);
    g = fma(-lds(118), lds(57), g);
    g = fma(-lds(119), lds(58), g);
    g = fma(-lds(121), lds(117), g);
    put_lds(122, g); }
  { double g = 0.0;
    g = fma(-0.1, b[72], g);
    g = g / d[15];
    put_lds(123, g); }
  { double g = 0.0;
    g = fma(-0.6, b[75], g);
    g = g / d[17];
    put_lds(124, g); }
  { double g = 0.0;
    g = fma(-1.0, b[11], g);
    g = g / d[21];
    put_lds(125, g); }
  { double g = 0.0;
    g = fma(-0.07, b[73], g);
    g = fma(-lds(125), lds(56), g);
    g = g / d[22];
    put_lds(126, g); }
  { double g = 0.0;
    g = fma(-1.0, b[0], g);
    g = g / d[29];
    put_lds(127, g); }
  { double g = 0.0;
    g = fma(-0.15, b[74], g);
    g = fma(-lds(127), lds(116), g);
    g = g / d[30];
    put_lds(128, g); }
  { double g = 0.0;
    g = fma(1.0, b[1], g);
    g = fma(1.0, b[2], g);
    g = fma(1.0, b[3], g);
    g = fma(1.0, b[4], g);
    g = fma(1.0, b[5], g);
    g = fma(1.0, b[6], g);
    g = fma(1.0, b[7], g);
    g = fma(1.0, b[8], g);
    g = fma(1.0, b[9], g);
    g = fma(1.0, b[12], g);
    g = fma(1.0, b[71], g);
    g = g + diag; bad = bad || fabs(g) < DBL_MIN;
    g = fma(-lds(123), lds(45), g);
    g = fma(-lds(124), lds(47), g);
    g = fma(-lds(125), lds(57), g);
    g = fma(-lds(126), lds(58), g);
    g = fma(-lds(127), lds(117), g);
    g = fma(-lds(128), lds(122), g);
    d[31] = g; }
  return bad;
}
template <class LG>
__device__ __forceinline__ void solve(const double (&d)[32], LG lds, double (&x)[32]) {
  x[18] = fma(-lds(48), x[14], x[18]);
  x[19] = fma(-lds(51), x[18], x[19]);
  x[21] = fma(-lds(55), x[15], x[21]);
  x[23] = fma(-lds(59), x[16], x[23]);
  x[25] = fma(-lds(63), x[23], x[25]);
  x[25] = fma(-lds(64), x[24], x[25]);
  x[26] = fma(-lds(66), x[7], x[26]);
  x[26] = fma(-lds(67), x[8], x[26]);
  x[26] = fma(-lds(68), x[9], x[26]);
  x[26] = fma(-lds(69), x[16], x[26]);
  x[26] = fma(-lds(70), x[23], x[26]);
  x[26] = fma(-lds(71), x[24], x[26]);
  x[26] = fma(-lds(72), x[25], x[26]);
  x[27] = fma(-lds(74), x[0], x[27]);
  x[27] = fma(-lds(75), x[7], x[27]);
  x[27] = fma(-lds(76), x[8], x[27]);
  x[27] = fma(-lds(77), x[9], x[27]);
  x[27] = fma(-lds(78), x[10], x[27]);
  x[27] = fma(-lds(79), x[11], x[27]);
  x[27] = fma(-lds(80), x[12], x[27]);
  x[27] = fma(-lds(81), x[13], x[27]);
  x[27] = fma(-lds(82), x[14], x[27]);
  x[27] = fma(-lds(83), x[15], x[27]);
  x[27] = fma(-lds(84), x[16], x[27]);
  x[27] = fma(-lds(85), x[17], x[27]);
  x[27] = fma(-lds(86), x[19], x[27]);
  x[27] = fma(-lds(87), x[20], x[27]);
  x[27] = fma(-lds(88), x[22], x[27]);
  x[27] = fma(-lds(89), x[24], x[27]);
  x[27] = fma(-lds(90), x[25], x[27]);
  x[27] = fma(-lds(91), x[26], x[27]);
  x[28] = fma(-lds(96), x[10], x[28]);
  x[28] = fma(-lds(97), x[11], x[28]);
  x[28] = fma(-lds(98), x[14], x[28]);
  x[28] = fma(-lds(99), x[18], x[28]);
  x[28] = fma(-lds(100), x[20], x[28]);
  x[28] = fma(-lds(101), x[25], x[28]);
  x[28] = fma(-lds(102), x[26], x[28]);
  x[29] = fma(-lds(105), x[12], x[29]);
  x[29] = fma(-lds(106), x[13], x[29]);
  x[29] = fma(-lds(107), x[17], x[29]);
  x[29] = fma(-lds(108), x[19], x[29]);
  x[29] = fma(-lds(109), x[20], x[29]);
  x[29] = fma(-lds(110), x[22], x[29]);
  x[29] = fma(-lds(111), x[24], x[29]);
  x[29] = fma(-lds(112), x[25], x[29]);
  x[29] = fma(-lds(113), x[26], x[29]);
  x[29] = fma(-lds(114), x[27], x[29]);
  x[29] = fma(-lds(115), x[28], x[29]);
  x[30] = fma(-lds(118), x[21], x[30]);
  x[30] = fma(-lds(119), x[22], x[30]);
  x[30] = fma(-lds(120), x[28], x[30]);
  x[30] = fma(-lds(121), x[29], x[30]);
  x[31] = fma(-lds(123), x[15], x[31]);
  x[31] = fma(-lds(124), x[17], x[31]);
  x[31] = fma(-lds(125), x[21], x[31]);
  x[31] = fma(-lds(126), x[22], x[31]);
  x[31] = fma(-lds(127), x[29], x[31]);
  x[31] = fma(-lds(128), x[30], x[31]);
  x[31] = x[31] / d[31];
  x[30] = fma(-lds(122), x[31], x[30]);
  x[30] = x[30] / d[30];
  x[29] = fma(-lds(116), x[30], x[29]);
  x[29] = fma(-lds(117), x[31], x[29]);
  x[29] = x[29] / d[29];
  x[28] = fma(-lds(103), x[29], x[28]);
  x[28] = fma(-lds(104), x[30], x[28]);
  x[28] = x[28] / d[28];
  x[27] = fma(-lds(92), x[28], x[27]);
  x[27] = fma(-lds(93), x[29], x[27]);
  x[27] = fma(-lds(94), x[30], x[27]);
  x[27] = fma(-lds(95), x[31], x[27]);
  x[27] = x[27] / d[27];
  x[26] = fma(-lds(73), x[29], x[26]);
  x[26] = x[26] / d[26];
  x[25] = fma(-lds(65), x[26], x[25]);
  x[25] = x[25] / d[25];
  x[24] = fma(-lds(62), x[26], x[24]);
  x[24] = x[24] / d[24];
  x[23] = fma(-lds(60), x[24], x[23]);
  x[23] = fma(-lds(61), x[26], x[23]);
  x[23] = x[23] / d[23];
  x[22] = fma(-lds(58), x[31], x[22]);
  x[22] = x[22] / d[22];
  x[21] = fma(-lds(56), x[22], x[21]);
  x[21] = fma(-lds(57), x[31], x[21]);
  x[21] = x[21] / d[21];
  x[20] = fma(-lds(54), x[28], x[20]);
  x[20] = x[20] / d[20];
  x[19] = fma(-lds(52), x[20], x[19]);
  x[19] = fma(-lds(53), x[28], x[19]);
  x[19] = x[19] / d[19];
  x[18] = fma(-lds(49), x[20], x[18]);
  x[18] = fma(-lds(50), x[28], x[18]);
  x[18] = x[18] / d[18];
  x[17] = fma(-lds(47), x[31], x[17]);
  x[17] = x[17] / d[17];
  x[16] = fma(-lds(46), x[26], x[16]);
  x[16] = x[16] / d[16];
  x[15] = fma(-lds(45), x[31], x[15]);
  x[15] = x[15] / d[15];
  x[14] = fma(-lds(44), x[28], x[14]);
  x[14] = x[14] / d[14];
  x[13] = fma(-lds(43), x[31], x[13]);
  x[13] = x[13] / d[13];
  x[12] = fma(-lds(42), x[31], x[12]);
  x[12] = x[12] / d[12];
  x[11] = fma(-lds(41), x[28], x[11]);
  x[11] = x[11] / d[11];
  x[10] = fma(-lds(40), x[28], x[10]);
  x[10] = x[10] / d[10];
  x[9] = fma(-lds(39), x[26], x[9]);
  x[9] = x[9] / d[9];
  x[8] = fma(-lds(38), x[26], x[8]);
  x[8] = x[8] / d[8];
  x[7] = fma(-lds(37), x[26], x[7]);
  x[7] = x[7] / d[7];
  x[6] = fma(-lds(36), x[29], x[6]);
  x[6] = x[6] / d[6];
  x[5] = fma(-lds(33), x[25], x[5]);
  x[5] = fma(-lds(34), x[29], x[5]);
  x[5] = fma(-lds(35), x[30], x[5]);
  x[5] = x[5] / d[5];
  x[4] = fma(-lds(31), x[28], x[4]);
  x[4] = fma(-lds(32), x[29], x[4]);
  x[4] = x[4] / d[4];
  x[3] = fma(-lds(18), x[12], x[3]);
  x[3] = fma(-lds(19), x[13], x[3]);
  x[3] = fma(-lds(20), x[17], x[3]);
  x[3] = fma(-lds(21), x[19], x[3]);
  x[3] = fma(-lds(22), x[20], x[3]);
  x[3] = fma(-lds(23), x[22], x[3]);
  x[3] = fma(-lds(24), x[24], x[3]);
  x[3] = fma(-lds(25), x[25], x[3]);
  x[3] = fma(-lds(26), x[26], x[3]);
  x[3] = fma(-lds(27), x[27], x[3]);
  x[3] = fma(-lds(28), x[28], x[3]);
  x[3] = fma(-lds(29), x[30], x[3]);
  x[3] = fma(-lds(30), x[31], x[3]);
  x[3] = x[3] / d[3];
  x[2] = fma(-lds(17), x[29], x[2]);
  x[2] = x[2] / d[2];
  x[1] = fma(-lds(0), x[7], x[1]);
  x[1] = fma(-lds(1), x[8], x[1]);
  x[1] = fma(-lds(2), x[9], x[1]);
  x[1] = fma(-lds(3), x[10], x[1]);
  x[1] = fma(-lds(4), x[11], x[1]);
  x[1] = fma(-lds(5), x[12], x[1]);
  x[1] = fma(-lds(6), x[13], x[1]);
  x[1] = fma(-lds(7), x[14], x[1]);
  x[1] = fma(-lds(8), x[15], x[1]);
  x[1] = fma(-lds(9), x[16], x[1]);
  x[1] = fma(-lds(10), x[17], x[1]);
  x[1] = fma(-lds(11), x[19], x[1]);
  x[1] = fma(-lds(12), x[20], x[1]);
  x[1] = fma(-lds(13), x[22], x[1]);
  x[1] = fma(-lds(14), x[24], x[1]);
  x[1] = fma(-lds(15), x[25], x[1]);
  x[1] = fma(-lds(16), x[30], x[1]);
  x[1] = x[1] / d[1];
  x[0] = x[0] / d[0];
}
}  // namespace unroll_Hg
