#include <hip/hip_runtime.h>
#include <cstdio>
#include <cmath>
__device__ unsigned rb(float f){unsigned u=__float_as_uint(f); if((u&0x7fffffff)>0x7f800000) return 0x7fc0; return (u+0x7fff+((u>>16)&1))>>16;}
// mismatches with the form of today and with a division, per constant
__global__ void go(unsigned* bad, unsigned* badd, unsigned* first, int nk){
  int x=blockIdx.x*256+threadIdx.x; if(x>=65536) return;
  float z=__uint_as_float((unsigned)x<<16);
  const float s=0x1p-24f;
  float d=fmaf(__expf(-z),s,s), r=__builtin_amdgcn_rcpf(d);
  unsigned a=rb(z*(s*fmaf(fmaf(-fminf(d,3e38f),r,1.0f),r,r)));
  unsigned b=rb(z/(1.0f+__expf(-z)));
  double zz=z; unsigned c=rb((float)(zz/(1.0+exp(-zz))));
  if(a!=b) atomicAdd(badd,1);
  if(b!=c) atomicAdd(badd+1,1);
  for(int k=0;k<nk;k++){
    float L=__uint_as_float(0x3fb8aa3bu+(k&15)-8);
    float one=s*(1.0f+0x1p-23f*((k>>4)&15)-0x1p-23f*8);
    float e=__builtin_amdgcn_exp2f(-z*L);
    float r2=__builtin_amdgcn_rcpf(fmaf(e,s,one));
    unsigned n=rb(z*(s*r2));
    if(n!=a){ atomicAdd(bad+k,1); first[k]=x; }
  }
}
int main(){
  unsigned*p; (void)hipMalloc(&p,4*(256*2+4)); (void)hipMemset(p,0,4*(256*2+4));
  go<<<256,256>>>(p,p+512,p+256,256);
  unsigned h[516]; (void)hipMemcpy(h,p,sizeof h,hipMemcpyDeviceToHost);
  printf("today vs division %u, division vs fp64 %u\n",h[512],h[513]);
  for(int k=0;k<256;k++) if(h[k]<3) printf("L %d one %d: %u (%04x)\n",(k&15)-8,(k>>4)-8,h[k],h[256+k]);
}
